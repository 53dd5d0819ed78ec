"""Values at the ends of the field (0 and P - 1), where the kernels' lazy sums
and products are largest or vanish, and query counts around the line (256, no
PoW) up to which the queries are drawn with the last mix. Against the oracle."""
import random

import numpy as np
import pytest

import pyoracle as po
import pyref_bytecode as pb
import vortexstark_amd as vx
from gpu_util import dev, empty, host, ptr
from test_gpu_bytecode import check
from vortexstark_amd import stwo
from vortexstark_amd._lib import call
import ctypes as C

pytestmark = pytest.mark.gpu
P = po.P


@pytest.mark.parametrize("log_n", [5, 14, 15, 24])  # one pass, one radix pass, generic and fixed shapes
@pytest.mark.parametrize("fill", ["zero", "high", "ends"])
def test_ntt(log_n, fill):
    print("ntt extremes", log_n, fill, flush=True)
    n, rng = 1 << log_n, np.random.default_rng(log_n)
    x = {"zero": lambda: np.zeros(n, np.uint32), "high": lambda: np.full(n, P - 1, np.uint32),
         "ends": lambda: rng.choice(np.array([0, P - 1], np.uint32), n)}[fill]()
    fwd, inv = po.stwo_twiddles(log_n)
    cache = stwo.StwoNttCache(log_n)
    d, e = dev(x), dev(x)
    call("vx_stwo_ntt_evaluate", ptr(d), C.c_void_p(cache.d_fwd_twiddles.as_ptr()), n, None)
    call("vx_stwo_ntt_interpolate", ptr(e), C.c_void_p(cache.d_inv_twiddles.as_ptr()), n, None)
    assert np.array_equal(host(d), po.stwo_evaluate(x, fwd, omp=True))
    assert np.array_equal(host(e), po.stwo_interpolate(x, inv, omp=True))


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("fill", ["zero", "high"])
def test_constraints(seed, fill):
    rng = random.Random(seed)
    prog = pb.random_program(rng, 40 + 60 * seed, 7, n_regs=24, offsets=(0, 1))
    value = P - 1 if fill == "high" else 0
    print("constraint extremes", seed, fill, prog.n_constraints(), flush=True)
    cols = [np.full(256, value, np.uint32) for _ in range(7)]
    coeff = [[value] * 4 for _ in range(prog.n_constraints())]
    acc = [np.full(256, value, np.uint32) for _ in range(4)]
    check(prog.encode(), cols, 256, 128, coeff, [P - 1, 1], acc)


@pytest.mark.parametrize("n_queries", [1, 255, 256, 257])
@pytest.mark.parametrize("pow_bits", [0, 4])
@pytest.mark.parametrize("graphs", [True, False])
def test_query_counts(n_queries, pow_bits, graphs):
    print("queries", n_queries, pow_bits, graphs, flush=True)
    p = vx.Prover(10, 2, n_queries, pow_bits, graphs=graphs)
    for a, b in ((3, 4), (P - 1, 0)):  # a second proof replays the graph
        assert p.prove(a, b) == po.prove(a, b, 10, n_queries=n_queries, pow_bits=pow_bits)
