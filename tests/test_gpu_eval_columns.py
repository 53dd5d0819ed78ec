"""vx_eval_at_point_batch and vx_oods_sample where the column table no longer
travels in the kernels' arguments (192 columns): one column below, at and
above it, and far above, sizes on both sides of the 2^14-coefficient chunk.
Against the oracle."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from gpu_util import dev, empty, host, ptr
from test_gpu_oods_chunks import run
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu
P = po.P


def sizes(n_cols):
    """Mostly tiny columns, a few of one and of four chunks, unsorted."""
    return [16 if k % 97 == 5 else 14 if k % 61 == 3 else (3 * k) % 7 for k in range(n_cols)]


@pytest.mark.parametrize("n_cols", [191, 192, 193, 2500])
def test_values(n_cols):
    print("eval columns", n_cols, flush=True)
    rng = np.random.default_rng(n_cols)
    logs, max_log = sizes(n_cols), 17  # no column is as large as the point's domain
    factors = rng.integers(0, P, 4 * max_log, dtype=np.uint32)
    cols = [rng.integers(0, P, 1 << L, dtype=np.uint32) for L in logs]
    got = run(cols, max_log, factors)  # its columns' own sizes
    for k, c in enumerate(cols):
        assert tuple(int(v) for v in got[k]) == po.eval_at_point_factors(c, factors[4 * (max_log - logs[k]):]), k


@pytest.mark.parametrize("n_cols", [192, 193, 700])
def test_oods(n_cols):
    print("oods columns", n_cols, flush=True)
    rng = np.random.default_rng(n_cols)
    logs = sizes(n_cols)
    cols = [rng.integers(0, P, 1 << L, dtype=np.uint32) for L in logs]
    ch = po.PyChannel()
    ch.mix_digest([n_cols, 2, 7, 1, 8, 2, 8, 1])
    words = lambda: np.concatenate([np.frombuffer(ch.state, np.uint32), [ch.c.n_draws]]).astype(np.uint32)
    bufs, d_ch, pts, vals = [dev(c) for c in cols], dev(words()), empty(16), empty(8 * n_cols)
    call("vx_oods_sample", ptr(d_ch), (C.c_void_p * n_cols)(*[b.ptr for b in bufs]), (C.c_uint32 * n_cols)(*logs), n_cols,
         9, ptr(pts), ptr(vals), None)
    want_pts, want_vals = ch.oods_sample(cols, 9)
    assert np.array_equal(host(pts), want_pts) and np.array_equal(host(vals), want_vals)
    assert np.array_equal(host(d_ch), words())
