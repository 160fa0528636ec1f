"""Instances of interval batches whose rounds in the LDS kernel (pcx_local.hip) keep
tightening many variables, more than a sixteenth as many as there are propagators:
after four such rounds they go on in full sweeps, beside others that stay.  Against
the oracle, and by the counts: one evaluation of the whole table a round."""
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


@pytest.mark.parametrize("n_inst", [2, 5, 700])
@pytest.mark.parametrize("mode", [pcx.MODE_PERSISTENT, pcx.MODE_BATCHED])
@pytest.mark.parametrize("chains,links", [(1, 70), (20, 30), (100, 41)])
def test_chains_that_rise_together(gpu, n_inst, mode, chains, links):
    """Precedence chains whose variables all rise by one a round; of five instances
    one fails at their end, one is empty, one is at its fixpoint and one rises along
    a single chain."""
    v = np.arange(chains * (links + 1), dtype=np.int32).reshape(chains, links + 1)
    V = v.size + 1
    x, y = v[:, 1:].reshape(-1), v[:, :-1].reshape(-1)
    P = x.size
    p = np.random.default_rng(chains).permutation(P)
    lb, ub = np.zeros(V, np.int32), np.full(V, 1000, np.int32)
    lb[V - 1] = ub[V - 1] = 1
    pir = pcx.PIR()
    pir.tell(np.full(P, ol.OPS["ADD"], np.int32), x[p], y[p], np.full(P, V - 1, np.int32), lb, ub)
    lo, hi = np.tile(lb, (n_inst, 1)), np.tile(ub, (n_inst, 1))
    for k in range(n_inst):
        if k % 5 == 1:
            hi[k, v[-1, -1]] = links - 1                      # fails
        elif k % 5 == 2:
            lo[k, 3], hi[k, 3] = 5, 4                         # empty
        elif k % 5 == 3:
            one_l, one_h = lb.copy(), ub.copy()
            ol.fixpoint(*pir.table(), one_l, one_h)
            lo[k], hi[k] = one_l, one_h                       # at its fixpoint
        elif k % 5 == 4:
            one_l, one_h = lb.copy(), ub.copy()
            ol.fixpoint(*pir.table(), one_l, one_h)
            lo[k], hi[k] = one_l, one_h
            lo[k, 0] = 7                                      # one chain rises
    want = [lo.reshape(-1).copy(), hi.reshape(-1).copy()]
    ro = ol.fixpoint_batch(*pir.table(), *want, V, threads=8)
    b = pcx.Batch(pir, n_inst, V)
    b.load(lo.reshape(-1), hi.reshape(-1))
    for _ in range(2):
        rg, st = b.run(mode)
        got = [a.reshape(n_inst, V) for a in b.read()]
        fo = np.array([r.failed for r in ro], bool)
        assert np.array_equal(rg.failed != 0, fo)
        assert all(np.array_equal(g[~fo], w.reshape(n_inst, V)[~fo]) for g, w in zip(got, want))
        assert np.array_equal((rg.has_changed != 0)[~fo], np.array([r.has_changed for r in ro], bool)[~fo])
        k = np.arange(n_inst) % 5
        if mode == pcx.MODE_PERSISTENT:
            assert (rg.evals[k == 0] == rg.sweeps[k == 0] * P).all()
            assert (rg.evals[k == 2] == 0).all() and (rg.evals[k == 3] == P).all()
        b.reset()
        assert all(np.array_equal(g, w.reshape(-1)) for g, w in zip(b.read(), (lo, hi)))


def test_subsets_and_one_store_by_itself(gpu):
    """The same over half of the table per instance, and a single store, which
    stays in the LDS kernel."""
    chains, links, n_inst = 20, 30, 6
    v = np.arange(chains * (links + 1), dtype=np.int32).reshape(chains, links + 1)
    V = v.size + 1
    x, y = v[:, 1:].reshape(-1), v[:, :-1].reshape(-1)
    P = x.size
    lb, ub = np.zeros(V, np.int32), np.full(V, 1000, np.int32)
    lb[V - 1] = ub[V - 1] = 1
    pir = pcx.PIR()
    pir.tell(np.full(P, ol.OPS["ADD"], np.int32), x, y, np.full(P, V - 1, np.int32), lb, ub)
    sub = [np.sort(np.random.default_rng(k).choice(P, P - 7 * k, replace=False)) for k in range(n_inst)]
    off = np.concatenate([[0], np.cumsum([len(s) for s in sub])]).astype(np.int64)
    idx = np.concatenate(sub).astype(np.int32)
    b = pcx.Batch(pir, n_inst, V, off, idx)
    b.load(np.tile(lb, n_inst), np.tile(ub, n_inst))
    rg, _ = b.run(pcx.MODE_PERSISTENT)
    lg, ug = (a.reshape(n_inst, V) for a in b.read())
    t = pir.table()
    for k in range(n_inst):
        lo, hi = lb.copy(), ub.copy()
        r = ol.fixpoint(*(a[sub[k]] for a in t), lo, hi)
        assert not r.failed and not rg.failed[k]
        assert np.array_equal(lg[k], lo) and np.array_equal(ug[k], hi)
    lo, hi = lb.copy(), ub.copy()
    ol.fixpoint(*t, lo, hi)
    l, u = lb.copy(), ub.copy()
    assert not pir.fixpoint(l, u).failed
    assert np.array_equal(l, lo) and np.array_equal(u, hi)
