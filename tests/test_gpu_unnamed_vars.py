"""Stores with variables past the last one that a propagator names: loads that differ there,
and branchings that split them, mark nothing for them and reach the oracle's fixpoints."""
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


@pytest.mark.parametrize("extra", [1, 2, 1025])
@pytest.mark.parametrize("bits", [False, True], ids=["intervals", "bits"])
@pytest.mark.parametrize("limit", [0, 60], ids=["drained", "swept"])
def test_unnamed_variables_mark_nothing(gpu, bits, extra, limit):
    links, n = 40, 6
    named = links + 2                            # a chain from variable 0, and the value 0
    V = named + extra
    x, y = np.arange(1, links + 1, dtype=np.int32), np.arange(links, dtype=np.int32)
    z = np.full(links, named - 1, np.int32)
    rows = [named, V - 1]                        # where instances 1 and 4 differ, and variable 0 in 5
    if bits:
        pir = pcx.BitsPIR(max_sweeps=limit)
        w = np.full(V, ol.word(range(6)), np.uint64)
        w[named - 1] = ol.word([0])
        pir.tell(np.full(links, ol.BITS_OPS["ADD"], np.int32), x, y, z, w)
        inst = np.tile(w, (n, 1))
        inst[1, rows[0]], inst[4, rows[1]], inst[5, 0] = ol.word([2]), ol.word([1, 4]), ol.word([3])
        stores = [inst.reshape(-1)]
    else:
        pir = pcx.PIR(max_sweeps=limit)
        lo, hi = np.zeros(V, np.int32), np.full(V, 9, np.int32)
        hi[named - 1] = 0
        pir.tell(np.full(links, ol.OPS["ADD"], np.int32), x, y, z, lo, hi)
        lb, ub = np.tile(lo, (n, 1)), np.tile(hi, (n, 1))
        ub[1, rows[0]], lb[4, rows[1]], ub[5, 0] = 3, 7, 0
        stores = [lb.reshape(-1), ub.reshape(-1)]

    def oracle(a):
        out = [s.copy() for s in a]
        run = ol.bits_fixpoint_batch if bits else ol.fixpoint_batch
        return out, run(*pir.table(), *out, V)

    def check(b, start):
        want, ro = oracle(start)
        rg, _ = b.run(pcx.MODE_BATCHED)
        assert [r.failed for r in rg] == [r.failed for r in ro]
        got = [b.read_words()] if bits else list(b.read())
        assert all((g == s).all() for g, s in zip(got, want))
        return got

    parent = pcx.Batch(pir, n, V)
    for _ in range(2):
        parent.load_words(*stores) if bits else parent.load(*stores)
        got = check(parent, stores)
    child = pcx.Batch(pir, 2 * n, V)             # instance 5's chain is fixed: it splits an unnamed variable
    var = parent.branch(child, from_fixpoint=True)
    assert var[5] == named and var[0] == 0
    start = [child.read_words()] if bits else list(child.read())
    check(child, start)
