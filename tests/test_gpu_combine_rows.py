"""Quotient combination around the row count (2^17) up to which a lane takes one
row, and around its workgroups of 256 and 2048 rows. Against the oracle."""
import numpy as np
import pytest

import pyoracle as po
from gpu_util import Pin, dev, empty, host, ptr, sync
from test_gpu_quotient_extremes import dev_ptrs, full
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rows", [255, 256, 257, 131071, 131072, 131073, 133120, 135170])
@pytest.mark.parametrize("fill", ["high", "zero", "random"])
def test_combine(n_rows, fill):
    print("combine rows", n_rows, fill, flush=True)
    rng = np.random.default_rng(n_rows)
    L = max(9, int(n_rows - 1).bit_length())
    logs = [L, L - 2, L]
    sx, sy, fla = (full(12, fill, rng) for _ in range(3))
    numers = [[full(1 << g, fill, rng) for _ in range(4)] for g in logs]
    xs, ys = full(n_rows, fill, rng), full(n_rows, fill, rng)
    nb = [[dev(c) for c in acc] for acc in numers]
    outs, pin = [empty(n_rows) for _ in range(4)], Pin()
    call("vx_compute_quotients_combine", pin(dev(sx)), pin(dev(sy)), pin(dev(fla)),
         *[pin(dev_ptrs([acc[k] for acc in nb])) for k in range(4)], pin(dev(np.array(logs, np.uint32))), 3,
         pin(dev(xs)), pin(dev(ys)), L, n_rows, *[ptr(o) for o in outs], None)
    sync()
    want = po.quotients_combine(sx, sy, fla, numers, logs, xs, ys, L)
    for k in range(4):
        assert np.array_equal(host(outs[k]), want[k]), k
