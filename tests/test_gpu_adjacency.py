"""The adjacency built on the device (pcx_adj.hip), through runs that evaluate a
propagator again only when the adjacency says so: a chain over variables in random
order stops at the first missing entry.  Variables around a scan's tile of 4,096
counts, tables around a wave and a workgroup, repeated operands, one variable in
every propagator, variables that none names."""
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


def _chain(n, V, rng):
    """n links v[i+1] = v[i] + one over V variables (the last of which no propagator
    names unless n + 2 == V), with a propagator of repeated operands beside each."""
    one = 0
    v = rng.permutation(V - 1 if n + 2 == V else V - 2)[:n + 1] + 1
    lb, ub = np.zeros(V, np.int32), np.full(V, 1 << 20, np.int32)
    lb[one] = ub[one] = 1
    lb[v[0]] = 3
    kind = rng.integers(0, 4, n)
    a, b = v[1:], v[:-1]
    op = np.concatenate([np.full(n, pcx.ADD), np.full(n, pcx.MAX)])
    x = np.concatenate([a, np.where(kind == 0, a, np.where(kind == 1, b, a))])
    y = np.concatenate([b, np.where(kind == 0, a, np.where(kind == 1, b, a))])     # max(a, a), max(b, b), ...
    z = np.concatenate([np.full(n, one), np.where(kind == 0, a, np.where(kind == 1, b, np.where(kind == 2, a, b)))])
    perm = rng.permutation(2 * n)
    return [c[perm].astype(np.int32) for c in (op, x, y, z)], lb, ub


def _tell(tell, lb, ub, **kw):
    pir = pcx.PIR(**kw)
    pir.tell(*tell, lb.copy(), ub.copy())
    return pir


def _check(pir, lb, ub, run):
    lo, hi = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo, hi)
    l, u, failed = run(pir, lb.copy(), ub.copy())
    assert not ro.failed and not failed
    assert np.array_equal(l, lo) and np.array_equal(u, hi)


def _single(pir, l, u):
    r = pir.fixpoint(l, u)
    return l, u, r.failed


def _marked(pir, l, u):
    b = pcx.Batch(pir, 1, len(l))
    b.load(l, u)
    r, _ = b.run(pcx.MODE_BATCHED)
    return (*b.read(), r.failed[0])


@pytest.mark.parametrize("n,V", [(1, 4), (31, 40), (32, 4095), (127, 4096), (128, 4097), (129, 8192), (2000, 2002),
                                 (4094, 4096), (4095, 4097), (8000, 8193), (3000, 12289)])
def test_lds_runs(gpu, n, V):
    rng = np.random.default_rng(n)
    tell, lb, ub = _chain(n, V, rng)
    pir = _tell(tell, lb, ub)
    _check(pir, lb, ub, _single)
    if n + 2 == V:
        return
    # told more: another table (every second link's variable below one that had no name)
    last = np.full(len(tell[1][::2]), V - 1, np.int32)
    pir.tell(np.full(len(last), pcx.LEQ), np.zeros(len(last), np.int32), tell[1][::2], last, lb, ub)
    _check(pir, lb, ub, _single)


@pytest.mark.parametrize("n,V", [(3000, 3002), (3000, 70000), (3000, 1 << 20)])
def test_marked_runs(gpu, n, V):
    """Marked sweeps over stores too large for LDS, hundreds of tiles among them."""
    tell, lb, ub = _chain(n, V, np.random.default_rng(n + V))
    _check(_tell(tell, lb, ub, event_driven=1, lockstep=0), lb, ub, _marked)
