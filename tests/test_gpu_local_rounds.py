"""How an instance of the LDS kernel (pcx_local.hip) starts and ends, against the
oracle: empty as loaded, failing in the first evaluations of its first round, or
at its fixpoint.  Rounds are counted from the first evaluation, so an instance that
is empty as loaded counts none and one that fails in its first round counts one."""
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


def _network(V, P):
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=11, nvars=V, nprops=P, chain_len=40))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    return pir, lb, ub


def _fails_at_once(pir, lb, ub):
    """Bounds with which the table's first propagators, one wave's share, all fail
    on their first evaluation: sums above what their operands allow."""
    top, tx, _, _ = pir.table()
    assert (top[:64] == pcx.ADD).all()
    lo, hi = lb.copy(), ub.copy()
    lo[tx[:64]] = hi[tx[:64]] = hi.max() * 2 + 1000000
    return lo, hi


@pytest.mark.parametrize("n_inst,mode", [(3, pcx.MODE_PERSISTENT), (12, pcx.MODE_BATCHED),
                                         (600, pcx.MODE_BATCHED), (2400, pcx.MODE_PERSISTENT)])
def test_instances_that_end_in_their_first_round(gpu, n_inst, mode):
    """Workgroups take one instance after another: those that fail at once, those
    that are empty as loaded and those that run to their fixpoint, in turn."""
    V, P = 500, 2001
    pir, lb, ub = _network(V, P)
    lo, hi = np.tile(lb, (n_inst, 1)), np.tile(ub, (n_inst, 1))
    lo[0::3], hi[0::3] = _fails_at_once(pir, lb, ub)
    lo[1::3, V - 1], hi[1::3, V - 1] = 5, 4
    lo_o, hi_o = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo_o, hi_o)
    b = pcx.Batch(pir, n_inst, V)
    b.load(lo.reshape(-1), hi.reshape(-1))
    res, _ = b.run(mode)
    failed = np.arange(n_inst) % 3 != 2
    assert not ro.failed and np.array_equal(res.failed != 0, failed)
    assert (res.sweeps[0::3] == 1).all() and (res.evals[0::3] == P).all()
    assert (res.sweeps[1::3] == 0).all() and (res.evals[1::3] == 0).all()
    assert (res.sweeps[2::3] > 1).all() and (res.has_changed[2::3] != 0).all()
    lg, ug = b.read()
    assert (lg.reshape(n_inst, V)[2::3] == lo_o).all() and (ug.reshape(n_inst, V)[2::3] == hi_o).all()


def test_single_stores_that_end_in_their_first_round(gpu):
    V, P = 4001, 16003
    pir, lb, ub = _network(V, P)
    for _ in range(3):
        lo, hi = _fails_at_once(pir, lb, ub)
        r = pir.fixpoint(lo, hi)
        assert r.failed and r.sweeps == 1 and r.evals == P
        lo, hi = lb.copy(), ub.copy()
        lo[V - 1], hi[V - 1] = 5, 4
        r = pir.fixpoint(lo, hi)
        assert r.failed and r.sweeps == 0 and r.evals == 0
