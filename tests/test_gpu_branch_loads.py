"""Batches that are by turns children of a branching (drained with an undo log) and
loaded batches whose first sweep is seeded (drained from lists of seeds, which lie in
the log's room): runs and resets against the oracle after each."""
import numpy as np
import pytest

import oracle_lib as ol
import pcx
from pcx.device import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


@pytest.mark.parametrize("first", ["load", "branch"])
@pytest.mark.parametrize("host", [False, True], ids=["device", "host"])
def test_loads_and_branchings_by_turns(gpu, first, host):
    V, P, n = 3001, 12007, 6
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=9, nvars=V, nprops=P, chain_len=30))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    assert not pir.fixpoint(lb, ub).failed
    lo, hi = pcx.gen_splits(10, lb, ub, 2 * n, 1, 20)
    parent, child = pcx.Batch(pir, n, V), pcx.Batch(pir, 2 * n, V)
    parent.load(np.tile(lb, n), np.tile(ub, n))
    parent.run(pcx.MODE_BATCHED)
    dev = DeviceArray(lo), DeviceArray(hi)

    def check(image):
        want = [a.copy() for a in image]
        ro = ol.fixpoint_batch(*pir.table(), *want, V, threads=4)
        for _ in range(2):
            rg, st = child.run(pcx.MODE_BATCHED)
            assert st.full_evals == 0                     # drained
            assert [bool(r.failed) for r in rg] == [bool(r.failed) for r in ro]
            ok = np.array([not r.failed for r in ro])
            for g, w in zip(child.read(), want):
                assert np.array_equal(g.reshape(2 * n, V)[ok], w.reshape(2 * n, V)[ok])
            child.reset()
            assert all(np.array_equal(g, w) for g, w in zip(child.read(), image))
            if image is not lists:                        # a branching's marks serve one run
                break

    lists = (lo, hi)
    for turn in range(4):
        if (turn + (first == "branch")) % 2:
            parent.branch(child, from_fixpoint=True)
            check(tuple(child.read()))
        else:
            if host:
                child.load(lo, hi)
            else:
                child.load_device(dev[0].ptr, dev[1].ptr)
            check(lists)
    for d in dev:
        d.close()
