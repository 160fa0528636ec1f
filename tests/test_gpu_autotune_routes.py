"""The autotuner over small stores: the event-driven LDS kernel is one of the points,
the engine keeps it for the batch when it wins, and single stores keep the kernels
that their own settings choose."""
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


def _engine(V, P):
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=21, nvars=V, nprops=P))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    return pir, lb, ub


def _fixpoint(pir, lb, ub):
    lo, hi = lb.copy(), ub.copy()
    assert not ol.fixpoint(*pir.table(), lo, hi).failed
    l, u = lb.copy(), ub.copy()
    r = pir.fixpoint(l, u)
    assert not r.failed and np.array_equal(l, lo) and np.array_equal(u, hi)
    return r


@pytest.mark.parametrize("subsets", [False, True], ids=["whole", "subsets"])
def test_small_stores(gpu, subsets):
    """200 links deep, 8,000 propagators: full sweeps do 25 times the evaluations of
    the event-driven kernel, which takes a third of the time or less."""
    V, P, n_inst = 2000, 8000, 64
    pir, lb, ub = _engine(V, P)
    before = _fixpoint(pir, lb, ub)
    lo, hi = pcx.gen_splits(22, lb, ub, n_inst, 1, 3)
    off, idx = pcx.gen_subsets(23, P, n_inst, 9 * P // 10, P) if subsets else (None, None)
    b = pcx.Batch(pir, n_inst, V, off, idx)
    b.load(lo, hi)
    best, points = b.autotune(reps=2)
    auto = [p for p in points if p["mode"] == pcx.MODE_PERSISTENT and p["lds_mode"] == 1 and p["event_driven"] == -1]
    assert len(auto) == 1 and all(p["ms"] > 0 for p in points)
    assert best == auto[0]
    lo_o, hi_o = lo.copy(), hi.copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, idx=idx.astype(np.int64) if subsets else None, off=off,
                           threads=8)
    res, _ = b.run(best["mode"])
    fo = np.array([r.failed for r in ro], bool)
    lg, ug = b.read()
    assert np.array_equal(res.failed != 0, fo)
    assert np.array_equal(lg.reshape(n_inst, V)[~fo], lo_o.reshape(n_inst, V)[~fo])
    assert np.array_equal(ug.reshape(n_inst, V)[~fo], hi_o.reshape(n_inst, V)[~fo])
    after = _fixpoint(pir, lb, ub)
    assert after.evals < 20 * P and before.evals < 20 * P  # not a full sweep a link
    pir2, _, _ = _engine(V, P)                             # the same point from a cache
    assert pcx.apply_tuning(pir2, best) == pcx.MODE_PERSISTENT
    assert _fixpoint(pir2, lb, ub).evals < 20 * P


def test_single_stores_beside_a_tuned_batch(gpu):
    """A batch whose stores do not fit in LDS is tuned to explicit settings; one store
    still chases: a handful of sweeps, not one a link."""
    V, P, n_inst = 24000, 96000, 3
    pir, lb, ub = _engine(V, P)
    before = _fixpoint(pir, lb, ub)
    b = pcx.Batch(pir, n_inst, V)
    b.load(np.tile(lb, n_inst), np.tile(ub, n_inst))
    best, _ = b.autotune(reps=1)
    assert pir.get_config().event_driven == best["event_driven"] != -1
    after = _fixpoint(pir, lb, ub)
    assert before.sweeps < 40 and after.sweeps < 40
