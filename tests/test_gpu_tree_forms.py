"""Trees of 8 and 16 leaves per lane on both sides of the line (512 workgroups)
where their hashing changes its form, every stored level against the oracle.
The shape is pinned through the tuner's cache file."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
import vortexstark_amd as vx
from gpu_util import dev, empty, host, ptr
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_log,lane_log,log_n", [(11, 3, 12), (11, 3, 19), (11, 3, 20), (12, 4, 13), (12, 4, 20),
                                                     (12, 4, 21)])
@pytest.mark.parametrize("n_cols", [1, 5])
def test_levels(tmp_path, tile_log, lane_log, log_n, n_cols):
    print("tree form", tile_log, lane_log, log_n, n_cols, flush=True)
    store_lo = lane_log + 3  # a key that no other test commits
    f = tmp_path / "tune.txt"
    f.write_text(f"0 {n_cols} 0 0 {log_n} {store_lo} {tile_log} {lane_log}\n")
    vx.tuner(True, str(f))
    try:
        rng = np.random.default_rng(log_n)
        cols = [rng.integers(0, po.P, 1 << log_n, dtype=np.uint32) for _ in range(n_cols)]
        bufs, root = [dev(c) for c in cols], empty(8)
        levels = empty(sum(8 << (log_n - k) for k in range(store_lo, log_n + 1)))
        call("vx_merkle_commit_tiled", (C.c_void_p * n_cols)(*[b.ptr for b in bufs]), n_cols, log_n, store_lo,
             ptr(levels), ptr(root), None)
        got, want, at = host(levels).reshape(-1, 8), po.leaf_hashes(cols), 0
        for level in range(1, log_n + 1):
            want = po.hash_nodes(want.reshape(-1))
            if level >= store_lo:
                assert np.array_equal(got[at:at + len(want)], want), level
                at += len(want)
        assert np.array_equal(host(root), want[0])
    finally:
        vx.tuner(True, None)
