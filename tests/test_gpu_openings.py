"""The decommitment's packing (two queries of a tree per wavefront, 16 lanes
per opening): odd query counts leave half a wavefront idle, the smallest
trees have fewer than 16 leaves per group, and next-row openings cross group
edges and wrap. Proof bytes against the oracle."""
import pytest

import pyoracle as po
import vortexstark_amd as vx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n,bb,nq", [(4, 1, 1), (4, 1, 3), (5, 2, 2), (9, 2, 81), (13, 1, 7)])
def test_fibonacci_openings(log_n, bb, nq):
    print("openings fib", log_n, bb, nq, flush=True)
    assert vx.Prover(log_n, bb, nq).prove(1, 5) == po.prove(1, 5, log_n, bb, nq)


@pytest.mark.parametrize("log_n,cols,nq", [(4, 34, 1), (4, 5, 255), (7, 16, 33)])
def test_next_row_openings(log_n, cols, nq):
    print("openings d2", log_n, cols, nq, flush=True)
    got = vx.D2Prover(log_n, cols, 4, 11, 1, nq).prove(77)
    assert got == po.d2_prove(77, log_n, cols, 4, 11, 1, nq, 0)


@pytest.mark.parametrize("logs,nq", [([14], 1), ([14] * 19, 5)])
def test_lifted_openings(logs, nq):
    print("openings lifted", logs, nq, flush=True)
    assert vx.BatchProver(logs, 1, nq).prove(9) == po.batch_prove(9, logs, 1, nq, 0)
