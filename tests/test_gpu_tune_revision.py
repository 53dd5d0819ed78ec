"""Choices saved by other kernels are not taken: a cache-file line carries the
revision of the kernels that were timed."""
import numpy as np
import pytest

import ctypes as C

import vortexstark_amd as vx
from gpu_util import dev, empty, ptr
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu


def entry(n_cols, log_n):
    return [e for e in vx.tuner_entries() if (e["leaf_kind"], e["n_cols"], e["log_n"], e["store_lo"]) == (0, n_cols, log_n, 5)]


def commit(n_cols, log_n):
    bufs = [dev(np.arange(1 << log_n, dtype=np.uint32)) for _ in range(n_cols)]
    levels, root = empty(sum(8 << (log_n - k) for k in range(5, log_n + 1))), empty(8)
    call("vx_merkle_commit_tiled", (C.c_void_p * n_cols)(*[b.ptr for b in bufs]), n_cols, log_n, 5, ptr(levels),
         ptr(root), None)


def test_lines_of_another_revision_are_measured_again(tmp_path):
    f = tmp_path / "tune.txt"
    try:
        vx.tuner(True, str(f))
        commit(13, 12)  # keys that no other test commits
        line = [ln.split() for ln in f.read_text().split("\n") if ln.startswith("0 13 0 0 12 5 ")]
        assert len(line) == 1 and len(line[0]) == 9 and line[0][8][0] == "r", line
        rev = int(line[0][8][1:])
        f.write_text(f"0 13 0 0 13 5 12 4 r{rev}\n0 13 0 0 14 5 12 4 r{rev + 1}\n0 13 0 0 15 5 12 4\n"
                     f"ntt 1 27 27 5 1 1 0 r{rev}\nntt 1 28 28 5 1 1 0 r{rev + 1}\nntt 1 29 29 5 1 1 0\n")
        vx.tuner(True, str(f))
        assert len(entry(13, 13)) == 1 and not entry(13, 14) and len(entry(13, 15)) == 1
        sizes = {e["log_n"] for e in vx.tuner_ntt_entries() if (e["n_cols"], e["stwo"]) == (5, True)}
        assert 27 in sizes and 28 not in sizes and 29 in sizes
        commit(13, 14)
        assert len(entry(13, 14)) == 1
        assert f.read_text().split("\n")[-2].split()[4:6] == ["14", "5"]
        assert f.read_text().split("\n")[-2].endswith(f"r{rev}")
    finally:
        vx.tuner(True, None)
