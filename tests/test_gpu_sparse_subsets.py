"""Persistent runs of batches whose subsets are a small, a middling or a large part
of the table: full sweeps of the subset below a third of the table, the LDS kernel
from there on, against the oracle bit for bit."""
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


@pytest.mark.parametrize("n_inst", [7, 400])
@pytest.mark.parametrize("size", [1, 100, 2000, 2001, 2002, 5000])
def test_persistent_subsets(gpu, n_inst, size):
    """6,003 propagators: a third is 2,001.  An instance that runs in the LDS kernel
    counts the evaluations of one full sweep and of its marks; full sweeps count
    whole sweeps only."""
    V, P = 1501, 6003
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=4, nvars=V, nprops=P, chain_len=40))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    lo, hi = pcx.gen_splits(5, lb, ub, n_inst, 1, 4)
    rng = np.random.default_rng(6)
    off = np.arange(n_inst + 1, dtype=np.int64) * size
    idx = np.concatenate([np.sort(rng.choice(P, size, replace=False)) for _ in range(n_inst)]).astype(np.int32)
    lo_o, hi_o = lo.copy(), hi.copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, idx=idx.astype(np.int64), off=off, threads=8)
    b = pcx.Batch(pir, n_inst, V, off, idx)
    b.load(lo, hi)
    rg, st = b.run(pcx.MODE_PERSISTENT)
    fo = np.array([r.failed for r in ro], bool)
    lg, ug = b.read()
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(lg.reshape(n_inst, V)[~fo], lo_o.reshape(n_inst, V)[~fo])
    assert np.array_equal(ug.reshape(n_inst, V)[~fo], hi_o.reshape(n_inst, V)[~fo])
    whole = bool((rg.evals == rg.sweeps * size).all())
    assert whole == (size < 2001) or size == 1
