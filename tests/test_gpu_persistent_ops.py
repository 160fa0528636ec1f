"""Full persistent sweeps (k_persistent, marks off) over tables of every opcode,
alone and together, against the oracle bit for bit: tables that end inside a wave
and around a workgroup's two propagators a lane, stores in LDS and in place."""
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


@pytest.mark.parametrize("lds", [0, 1])
@pytest.mark.parametrize("ops", [[o] for o in range(10)] + [[0, 1, 6, 7, 8, 9], list(range(10))],
                         ids=lambda ops: "-".join(map(str, ops)))
@pytest.mark.parametrize("P", [1, 63, 513, 1025, 1500])
def test_random_tables(gpu, ops, P, lds):
    rng = np.random.default_rng(100 * P + sum(ops))
    V0, n_inst = P // 2 + 4, 6
    V = V0 + P
    op = rng.choice(ops, P)
    y, z = rng.integers(0, V0, (2, P))
    x = V0 + np.arange(P)                                 # each result has its own variable
    w = np.concatenate([rng.integers(1, 40, V0), np.zeros(P, np.int64)])
    a, b = w[y], w[z]
    w[x] = np.choose(op, [a + b, a * b, a // b, a // b, -(-a // b), a // b, np.minimum(a, b), np.maximum(a, b),
                          (a == b) * 1, (a <= b) * 1])
    lb, ub = w - rng.integers(0, 4, V), w + rng.integers(0, 4, V)
    wide = rng.random(V) < 0.3
    lb[wide], ub[wide] = np.where(rng.random(wide.sum()) < 0.2, pcx.MINF, -50), 5000
    reified = x[op >= 8]
    lb[reified], ub[reified] = np.maximum(lb[reified], 0), np.minimum(ub[reified], 1)
    lb, ub = lb.astype(np.int32), ub.astype(np.int32)
    pir = pcx.PIR(event_driven=0, lds_mode=lds)
    pir.tell(op, x, y, z, lb, ub)
    lo, hi = np.tile(lb, (n_inst, 1)), np.tile(ub, (n_inst, 1))
    for k in range(1, n_inst):                            # the solution in some variables
        at = rng.integers(0, V, V // 8)
        lo[k, at] = hi[k, at] = w[at]
    lo[5, x[-1]] = hi[5, x[-1]] = w[x[-1]] + 2000         # no solution
    lo, hi = lo.reshape(-1), hi.reshape(-1)
    lo_o, hi_o = lo.copy(), hi.copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, threads=4)
    fo = np.array([r.failed for r in ro], bool)
    assert not fo[:5].any()
    batch = pcx.Batch(pir, n_inst, V)
    batch.load(lo, hi)
    rg, _ = batch.run(pcx.MODE_PERSISTENT)
    assert np.array_equal(rg.failed != 0, fo)
    lg, ug = batch.read()
    assert np.array_equal(lg.reshape(n_inst, V)[~fo], lo_o.reshape(n_inst, V)[~fo])
    assert np.array_equal(ug.reshape(n_inst, V)[~fo], hi_o.reshape(n_inst, V)[~fo])
    assert np.array_equal((rg.has_changed != 0)[~fo], np.array([r.has_changed for r in ro], bool)[~fo])
