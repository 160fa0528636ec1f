"""Networks with one variable that most propagators name (a makespan above every
task's end, an objective), which is tightened link after link: against the oracle
bit for bit, around the degree from which its neighbours are left to a sweep or a
round of the whole table."""
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


def _tasks(L, F):
    """Tasks 0..L, each a unit after the one before, and F others, all below the
    makespan (variable 1); variable 0 is one.  Every link raises the makespan."""
    s, o = 2, 3 + L
    tell = [(pcx.ADD, s + i + 1, s + i, 0) for i in range(L)]
    tell += [(pcx.LEQ, 0, s + i, 1) for i in range(L + 1)]
    tell += [(pcx.LEQ, 0, o + j, 1) for j in range(F)]
    n = 3 + L + F
    lb, ub = np.zeros(n, np.int32), np.full(n, 100000, np.int32)
    lb[0] = ub[0] = 1
    lb[s] = 5
    return tell, lb, ub


def _through(K, F):
    """c = M + 1, t = min(c, K), t <= M, and F others below M: the climb of M to K
    leads through the hub at every link."""
    n = 5 + F
    tell = [(pcx.ADD, 2, 1, 0), (pcx.MIN, 4, 2, 3), (pcx.LEQ, 0, 4, 1)]
    tell += [(pcx.LEQ, 0, 5 + j, 1) for j in range(F)]
    lb, ub = np.zeros(n, np.int32), np.full(n, 100000, np.int32)
    lb[0] = ub[0] = 1
    lb[3] = ub[3] = K
    return tell, lb, ub


def _told(tell, lb, ub, seed, **kw):
    """Told in a random order (the table is sorted by opcode only)."""
    perm = np.random.default_rng(seed).permutation(len(tell))
    pir = pcx.PIR(**kw)
    pir.tell(*(np.array([p[i] for p in tell], np.int32)[perm] for i in range(4)), lb.copy(), ub.copy())
    return pir


def _check(pir, lb, ub):
    lo, hi = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo, hi)
    l, u = lb.copy(), ub.copy()
    r = pir.fixpoint(l, u)
    d_lb, d_ub = DeviceArray(lb), DeviceArray(ub)
    rn = pir.fixpoint_noalloc(d_lb.ptr, d_ub.ptr, len(lb))
    for got, a, b in ((r, l, u), (rn, d_lb.read(), d_ub.read())):
        assert bool(got.failed) == bool(ro.failed)
        if not ro.failed:
            assert bool(got.has_changed) == bool(ro.has_changed)
            assert np.array_equal(a, lo) and np.array_equal(b, hi)
    d_lb.close()
    d_ub.close()
    return r


NETS = {"tasks": _tasks, "through": _through}


@pytest.mark.parametrize("net", NETS)
@pytest.mark.parametrize("F", [0, 100, 124, 125, 126, 127, 128, 129, 2000, 40000])
def test_chases(gpu, net, F):
    """Single stores in sweeps that chase: the hub's degree at, below and above 128
    and far above; and a makespan too low, which fails."""
    tell, lb, ub = NETS[net](60, F)
    pir = _told(tell, lb, ub, F, lds_mode=0)
    _check(pir, lb, ub)
    hi = ub.copy()
    hi[1] = 40
    assert _check(pir, lb, hi).failed
