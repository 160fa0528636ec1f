"""How many tightened variables a round of the LDS kernel (pcx_local.hip) lists and
walks before it evaluates every propagator instead: against the oracle, and by the
evaluations counted, on both sides of the line (a sixteenth of the propagators, at
least 64 and at most what the list holds)."""
import numpy as np
import pytest

import oracle_lib as ol
import pcx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


@pytest.mark.parametrize("n_inst", [3, 300])
@pytest.mark.parametrize("P,W,dense", [(300, 64, False), (300, 65, True), (1039, 64, False), (1040, 65, False),
                                       (1040, 66, True), (6400, 400, False), (6400, 401, True), (6400, 3000, True)])
def test_rounds_that_tighten_many(gpu, n_inst, P, W, dense):
    """Variable 0 bounds W leaves through one propagator each, in the first round;
    the second one finds nothing.  The other propagators bind nothing."""
    V = W + 3
    zero, free = W + 1, W + 2
    lo, hi = np.zeros(V, np.int32), np.full(V, 9, np.int32)
    hi[zero], hi[0] = 0, 5
    x = np.concatenate([1 + np.arange(W), np.full(P - W, free)]).astype(np.int32)
    y = np.concatenate([np.zeros(W), np.full(P - W, free)]).astype(np.int32)
    pir = pcx.PIR()
    pir.tell(np.full(P, ol.OPS["ADD"], np.int32), x, y, np.full(P, zero, np.int32), lo, hi)
    lb, ub = np.tile(lo, n_inst), np.tile(hi, n_inst)
    ub[0::V] = 3 + np.arange(n_inst) % 2
    want = [lb.copy(), ub.copy()]
    ro = ol.fixpoint_batch(*pir.table(), *want, V)
    b = pcx.Batch(pir, n_inst, V)
    b.load(lb, ub)
    rg, _ = b.run(pcx.MODE_PERSISTENT)
    assert not rg.failed.any() and not any(r.failed for r in ro)
    assert all(np.array_equal(g, w) for g, w in zip(b.read(), want))
    assert (rg.sweeps == 2).all() and (rg.evals == P + (P if dense else W)).all()
