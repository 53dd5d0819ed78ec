"""Size checks of the lifted leaf entry points, made on the host before
anything is allocated or launched."""
import ctypes as C

import pytest

from vortexstark_amd._lib import load

ARG = 1  # the status of an invalid argument


@pytest.mark.parametrize("n_cols", [1, 2, 128, 129])  # either side of the columns that travel in kernel arguments
@pytest.mark.parametrize("lifting_log", [0, 1, 32])
def test_leaves_refuse_trees_outside_2_to_31(n_cols, lifting_log):
    cols = (C.c_void_p * n_cols)(*[1 << 20] * n_cols)  # never read: the size is refused first
    logs = (C.c_uint32 * n_cols)(*[min(lifting_log, 1)] * n_cols)
    out = C.c_void_p(1 << 20)
    assert load().vx_build_leaves_lifted(cols, logs, n_cols, lifting_log, out, None) == ARG
