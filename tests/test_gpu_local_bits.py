"""Bitset batches in persistent mode on both sides of the rule that gives them to the
LDS kernel (12,288 propagators, or stores near their fixpoints): against the oracle,
and by the evaluations counted: full sweeps count whole sweeps."""
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
@pytest.mark.parametrize("P,root,local", [(3001, False, False), (12287, False, False), (12288, False, True),
                                          (12288, True, True), (8000, True, True)])
def test_persistent_bitsets(gpu, n_inst, P, root, local):
    V = P // 4
    op, x, y, z, words = pcx.gen_bits_network(5, V, P)
    pir = pcx.BitsPIR()
    pir.tell(op, x, y, z, words)
    if root:
        pir.fixpoint(words)
    w = pcx.gen_bits_splits(6, words, n_inst, 1, 6)
    w.reshape(n_inst, V)[1, 5] = 0                        # empty as loaded
    wo = w.copy()
    ro = ol.bits_fixpoint_batch(*pir.table(), wo, V, threads=8)
    b = pcx.Batch(pir, n_inst, V)
    b.load_words(w)
    rg, st = b.run(pcx.MODE_PERSISTENT)
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(b.read_words().reshape(n_inst, V)[~fo], wo.reshape(n_inst, V)[~fo])
    assert np.array_equal((rg.has_changed != 0)[~fo], np.array([r.has_changed for r in ro], bool)[~fo])
    assert bool((rg.evals == rg.sweeps * P).all()) == (not local)
