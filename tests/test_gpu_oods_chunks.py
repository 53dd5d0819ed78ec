"""The chunked evaluation of many columns (vx_eval_at_point_batch): more
columns than the kernels' arguments take, sizes around the 2^14-coefficient chunk,
several chunks per workgroup, and extreme coefficients (0 and P - 1, where
the 64-bit sums are largest). Field values against the oracle."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from gpu_util import dev, empty, host, ptr
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu
P = po.P


def run(cols, max_log, factors):
    bufs = [dev(c) for c in cols]
    out, f = empty(4 * len(cols)), dev(factors)
    call("vx_eval_at_point_batch", (C.c_void_p * len(cols))(*[b.ptr for b in bufs]),
         (C.c_uint32 * len(cols))(*[int(c.size).bit_length() - 1 for c in cols]), len(cols), ptr(f), max_log, ptr(out),
         None)
    return host(out).reshape(-1, 4)


@pytest.mark.parametrize("logs", [[0, 1, 2, 3, 5] * 79, [13, 14, 15, 16], [18] * 5 + [3], [26, 14, 26]])
@pytest.mark.parametrize("fill", ["random", "low", "high"])
def test_chunks_match_oracle(logs, fill):
    print("eval chunks", len(logs), max(logs), fill, flush=True)
    rng = np.random.default_rng(len(logs))
    max_log = max(logs)
    factors = rng.integers(0, P, 4 * max_log, dtype=np.uint32)
    if fill == "high":
        factors[:] = P - 1
    make = {"random": lambda n: rng.integers(0, P, n, dtype=np.uint32), "low": lambda n: np.zeros(n, np.uint32),
            "high": lambda n: np.full(n, P - 1, np.uint32)}[fill]
    cols = [make(1 << L) for L in logs]
    got = run(cols, max_log, factors)
    seen = {}
    for k, c in enumerate(cols):
        L = logs[k]
        key = L if fill != "random" else k
        if key not in seen:  # equal columns have equal values
            # a smaller column takes the last L factors
            seen[key] = po.eval_at_point_factors(c, factors[4 * (max_log - L):])
        assert tuple(int(v) for v in got[k]) == seen[key], (k, L)


@pytest.mark.parametrize("n_cols", [1, 2, 3, 127, 128, 129, 255])
def test_mixed_values(n_cols):
    """The transcript's message at the edges of its blocks (16 words) and of
    the 64 blocks laid out at a time (127 columns are 64 blocks)."""
    print("oods mix", n_cols, flush=True)
    rng = np.random.default_rng(n_cols)
    cols = [rng.integers(0, P, 8, dtype=np.uint32) for _ in range(n_cols)]
    ch = po.PyChannel()
    ch.mix_digest([n_cols, 2, 7, 1, 8, 2, 8, 1])
    words = lambda: np.concatenate([np.frombuffer(ch.state, np.uint32), [ch.c.n_draws]]).astype(np.uint32)
    bufs, d_ch, pts, vals = [dev(c) for c in cols], dev(words()), empty(16), empty(8 * n_cols)
    call("vx_oods_sample", ptr(d_ch), (C.c_void_p * n_cols)(*[b.ptr for b in bufs]), (C.c_uint32 * n_cols)(*[3] * n_cols),
         n_cols, 5, ptr(pts), ptr(vals), None)
    want_pts, want_vals = ch.oods_sample(cols, 5)
    assert np.array_equal(host(pts), want_pts) and np.array_equal(host(vals), want_vals)
    assert np.array_equal(host(d_ch), words())
