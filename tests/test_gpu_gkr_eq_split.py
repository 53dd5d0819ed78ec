"""The one-launch eq table where its split over lanes, values per lane and
workgroups changes: 2^8 lanes, one value per lane up to 2^17 entries, 32 from
2^22, with extreme coordinates. Against the oracle."""
import numpy as np
import pytest

import pyoracle as po
from gpu_util import dev, empty, host, ptr
from vortexstark_amd._lib import call

pytestmark = pytest.mark.gpu
P = po.P


@pytest.mark.parametrize("k", [2, 7, 8, 9, 15, 17, 18, 21, 22, 23])
@pytest.mark.parametrize("fill", ["random", "extreme"])
def test_eq_table(k, fill):
    print("gkr eq split", k, fill, flush=True)
    rng = np.random.default_rng(k)
    y, v = rng.integers(0, P, 4 * k, dtype=np.uint32), rng.integers(0, P, 4, dtype=np.uint32)
    if fill == "extreme":
        y = rng.choice(np.array([0, 1, P - 1], np.uint32), 4 * k)
        v[:] = P - 1
    out, dy, dv = empty(4 << k), dev(y), dev(v)
    call("vx_gkr_gen_eq_evals", ptr(out), ptr(dy), k, ptr(dv), None)
    assert np.array_equal(host(out), po.gkr_gen_eq_evals(y, v))
