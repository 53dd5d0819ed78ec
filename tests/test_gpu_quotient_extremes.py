"""Numerators and their combination where the kernels' 64-bit sums are largest
(every value P - 1) and where they vanish, at column counts around the step of
four and row counts around 2048 (one row per lane; test_gpu_combine_rows has
the counts around workgroups of eight rows per lane). Against the oracle."""
import numpy as np
import pytest

import pyoracle as po
from gpu_util import Pin, dev, empty, host, ptr, sync
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu
P = po.P


def dev_ptrs(bufs):
    return dev(np.array([b.ptr for b in bufs], np.uint64).view(np.uint32))


def full(n, fill, rng):
    return {"high": lambda: np.full(n, P - 1, np.uint32), "zero": lambda: np.zeros(n, np.uint32),
            "random": lambda: rng.integers(0, P, n, dtype=np.uint32)}[fill]()


@pytest.mark.parametrize("n_cols", [1, 3, 4, 5, 33])
@pytest.mark.parametrize("fill", ["high", "zero"])
def test_numerators(n_cols, fill):
    print("numerators", n_cols, fill, flush=True)
    n_rows = 1028
    col, coeff = full(n_rows, fill, None), full(4 * n_cols, fill, None)
    buf, outs, pin = dev(col), [empty(n_rows) for _ in range(8)], Pin()
    idx = np.arange(n_cols, dtype=np.uint32)
    call("vx_accumulate_numerators_dual", pin(dev_ptrs([buf] * n_cols)), pin(dev(idx)), pin(dev(idx)),
         *[pin(dev(coeff)) for _ in range(4)], n_cols, n_rows, *[ptr(o) for o in outs], None)
    sync()
    want = po.accumulate_numerators([col] * n_cols, list(idx), coeff, coeff, n_rows)
    for k in range(8):
        assert np.array_equal(host(outs[k]), want[k % 4]), k


@pytest.mark.parametrize("n_rows", [1, 2047, 2048, 2049])
@pytest.mark.parametrize("fill", ["high", "zero", "random"])
def test_combine(n_rows, fill):
    print("combine", n_rows, fill, flush=True)
    rng = np.random.default_rng(n_rows)
    L, logs = 12, [12, 10]
    sx, sy, fla = (full(8, fill, rng) for _ in range(3))
    numers = [[full(1 << g, fill, rng) for _ in range(4)] for g in logs]
    xs, ys = full(n_rows, fill, rng), full(n_rows, fill, rng)
    nb = [[dev(c) for c in acc] for acc in numers]
    outs, pin = [empty(n_rows) for _ in range(4)], Pin()
    call("vx_compute_quotients_combine", pin(dev(sx)), pin(dev(sy)), pin(dev(fla)),
         *[pin(dev_ptrs([acc[k] for acc in nb])) for k in range(4)], pin(dev(np.array(logs, np.uint32))), 2,
         pin(dev(xs)), pin(dev(ys)), L, n_rows, *[ptr(o) for o in outs], None)
    sync()
    want = po.quotients_combine(sx, sy, fla, numers, logs, xs, ys, L)
    for k in range(4):
        assert np.array_equal(host(outs[k]), want[k]), k
