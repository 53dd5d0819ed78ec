"""Batches at the line where column addresses no longer travel in a kernel's
arguments (128 columns): transforms, LDE and lifted leaves one column below, at
and above it, and leaf and node hashing around the size where the kernels
change their form (512 workgroups of 256). Against the oracle."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from gpu_util import dev, empty, host, ptr
from vortexstark_amd import stwo
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu
P = po.P


def ptrs(bufs):
    return (C.c_void_p * len(bufs))(*[b.ptr for b in bufs])


def addr(buf):
    return C.c_void_p(int(buf.as_ptr()))


@pytest.mark.parametrize("n_cols", [1, 127, 128, 129, 300])
@pytest.mark.parametrize("log_n", [5, 15])  # one pass; a strided and a contiguous pass
def test_batches(n_cols, log_n):
    print("column batch", n_cols, log_n, flush=True)
    rng = np.random.default_rng(n_cols)
    n, big = 1 << log_n, 2 << log_n
    cols = [rng.integers(0, P, n, dtype=np.uint32) for _ in range(n_cols)]
    cols[-1][:] = P - 1
    small, large = stwo.StwoNttCache(log_n), stwo.StwoNttCache(log_n + 1)
    values, evals = [dev(c) for c in cols], [empty(big) for _ in cols]
    call("vx_stwo_ntt_batch_interpolate", ptrs(values), addr(small.d_inv_twiddles), n, n_cols, None)
    call("vx_stwo_ntt_evaluate_lde_batch", ptrs(evals), ptrs(values), n, n_cols, addr(large.d_fwd_twiddles), big,
         None)
    back = [dev(host(v)) for v in values]
    call("vx_stwo_ntt_batch_evaluate", ptrs(back), addr(small.d_fwd_twiddles), n, n_cols, None)
    inv, fwd = po.stwo_twiddles(log_n)[1], po.stwo_twiddles(log_n + 1)[0]
    for k in sorted({0, n_cols // 2, n_cols - 1}):
        coeffs = po.stwo_interpolate(cols[k], inv)
        assert np.array_equal(host(values[k]), coeffs), k
        padded = np.concatenate([coeffs, np.zeros(n, np.uint32)])
        assert np.array_equal(host(evals[k]), po.stwo_evaluate(padded, fwd)), k
    for k, b in enumerate(back):
        assert np.array_equal(host(b), cols[k]), k


@pytest.mark.parametrize("n_cols,log_n", [(127, 8), (128, 8), (129, 8), (3, 16), (3, 17)])
def test_lifted_leaves(n_cols, log_n):
    print("lifted leaves", n_cols, log_n, flush=True)
    rng = np.random.default_rng(n_cols)
    logs = sorted([log_n] + [int(v) for v in rng.integers(log_n - 4, log_n + 1, n_cols - 1)])
    cols = [rng.integers(0, P, 1 << L, dtype=np.uint32) for L in logs]
    bufs, out = [dev(c) for c in cols], empty(8 << log_n)
    call("vx_build_leaves_lifted", ptrs(bufs), (C.c_uint32 * n_cols)(*logs), n_cols, log_n, ptr(out), None)
    assert np.array_equal(host(out).reshape(-1, 8), po.leaves_lifted(cols, log_n))


@pytest.mark.parametrize("n_cols,n", [(1, 131071), (4, 131072), (7, 131073), (16, 131328)])
def test_leaf_and_node_hashes(n_cols, n):
    print("leaf and node hashes", n_cols, n, flush=True)
    rng = np.random.default_rng(n)
    cols = [rng.integers(0, P, n, dtype=np.uint32) for _ in range(n_cols)]
    bufs, out = [dev(c) for c in cols], empty(8 * n)
    call("vx_merkle_hash_leaves_host", ptrs(bufs), ptr(out), n_cols, n, None)
    assert np.array_equal(host(out).reshape(-1, 8), po.leaf_hashes(cols))
    children = rng.integers(0, 1 << 32, 16 * n, dtype=np.uint32)
    par, ch = empty(8 * n), dev(children)
    call("vx_merkle_hash_nodes", ptr(ch), ptr(par), n, None)
    assert np.array_equal(host(par).reshape(-1, 8), po.hash_nodes(children))
