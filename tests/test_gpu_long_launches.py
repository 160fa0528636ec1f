"""Stores that converge slowly: a pair of variables that raise each other by one,
link after link, which no launch may follow for as long as it goes on.  Against the
oracle bit for bit, on networks of a handful of propagators."""
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


def _climb(c, top=1 << 30):
    """x = y + 1, t = min(x, c), t <= y: y climbs by one every three links from 0
    to c, where it stays (or fails, above `top`).  Variables: 0 is one, 1 y, 2 x,
    3 c, 4 t."""
    tell = [(pcx.ADD, 2, 1, 0), (pcx.MIN, 4, 2, 3), (pcx.LEQ, 0, 4, 1)]
    lb = np.array([1, 0, 0, c, 0], np.int32)
    ub = np.array([1, top, top, c, top], np.int32)
    return tell, lb, ub


def _told(tell, lb, ub, **kw):
    pir = pcx.PIR(**kw)
    pir.tell(*(np.array([p[i] for p in tell], np.int32) for i in range(4)), lb.copy(), ub.copy())
    return pir


def _same(pir, r, l, u, lb, ub):
    lo, hi = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo, hi)
    assert bool(r.failed) == bool(ro.failed)
    if not ro.failed:
        assert bool(r.has_changed) == bool(ro.has_changed)
        assert np.array_equal(l, lo) and np.array_equal(u, hi)


@pytest.mark.parametrize("c,top", [(200, 1 << 30), (20000, 1 << 30), (20000, 19000)])
def test_a_chase_ends_its_launch(gpu, c, top):
    """60,000 links in launches of at most 4,096 steps a wave.  The three propagators
    are one wave's; a step raises y by one at most (its lanes may hold all three, so it
    may be three links), after four plain sweeps."""
    tell, lb, ub = _climb(c, top)
    pir = _told(tell, lb, ub, lds_mode=0)
    l, u = lb.copy(), ub.copy()
    r = pir.fixpoint(l, u)
    _same(pir, r, l, u, lb, ub)
    assert r.evals > c
    d_lb, d_ub = DeviceArray(lb), DeviceArray(ub)
    rn = pir.fixpoint_noalloc(d_lb.ptr, d_ub.ptr, len(lb))
    _same(pir, rn, d_lb.read(), d_ub.read(), lb, ub)
    d_lb.close()
    d_ub.close()
    b = pcx.Batch(pir, 1, len(lb))
    b.load(lb, ub)
    rb, st = b.run(pcx.MODE_PLAIN)
    l, u = b.read()
    _same(pir, rb[0], l, u, lb, ub)
    if c > 10000:
        assert st.kernel_launches >= 4 + min(c, top) // 4096


def test_a_chase_leaves_a_failed_store(gpu):
    """One wave climbs without an end in sight (a step of y every three links) while
    others chase a chain of 300 links whose last one fails: the climb stops then, near
    y = 100, and not after its 4,096 links, beyond y = 1,365."""
    tell, lb, ub = _climb(1 << 29)
    L, n = 300, 5
    idle = list(range(n, n + 3 * 256))                   # propagators of other waves, with nothing to do
    tell += [(pcx.ADD, v, v + 1, v + 2) for v in idle[::3]]
    lb, ub = np.append(lb, np.tile([0, 0, 0], 256)), np.append(ub, np.tile([2, 1, 1], 256))
    s = len(lb)
    tell += [(pcx.ADD, s + i + 1, s + i, 0) for i in range(L)]
    lb, ub = np.append(lb, [7] + [0] * L).astype(np.int32), np.append(ub, [7] + [1 << 20] * L).astype(np.int32)
    ub[s + L] = 7 + L - 1
    pir = _told(tell, lb, ub, lds_mode=0)
    l, u = lb.copy(), ub.copy()
    r = pir.fixpoint(l, u)
    assert r.failed and l[1] < 1000


@pytest.mark.parametrize("c,top", [(200, 1 << 30), (20000, 1 << 30), (20000, 19000)])
def test_a_single_store_in_lds_takes_several_launches(gpu, c, top):
    """The LDS kernel on one store, in host memory and in the caller's device arrays;
    counts go on from launch to launch (a step raises y by one at most)."""
    tell, lb, ub = _climb(c, top)
    pir = _told(tell, lb, ub)
    l, u = lb.copy(), ub.copy()
    r = pir.fixpoint(l, u)
    _same(pir, r, l, u, lb, ub)
    assert r.sweeps >= min(c, top) and r.evals >= 3 * (min(c, top) - 1)
    d_lb, d_ub = DeviceArray(lb), DeviceArray(ub)
    rn = pir.fixpoint_noalloc(d_lb.ptr, d_ub.ptr, len(lb))
    _same(pir, rn, d_lb.read(), d_ub.read(), lb, ub)
    assert rn.sweeps >= min(c, top) and rn.evals >= 3 * (min(c, top) - 1)
    d_lb.close()
    d_ub.close()


@pytest.mark.parametrize("n_inst,mode", [(1, pcx.MODE_PLAIN), (1, pcx.MODE_BATCHED), (5, pcx.MODE_BATCHED),
                                         (5, pcx.MODE_PERSISTENT), (700, pcx.MODE_BATCHED),
                                         (700, pcx.MODE_PERSISTENT)])
def test_batches_in_lds_take_several_launches(gpu, n_inst, mode):
    """Instances that are done in the first launch (at their fixpoint, failed, empty
    as loaded) beside some that need four and one that fails in its third: each
    settled one keeps its store and its counts."""
    tell, lb, ub = _climb(12000)
    V = len(lb)
    pir = _told(tell, lb, ub, base_seed=0)
    lo, hi = np.tile(lb, (n_inst, 1)), np.tile(ub, (n_inst, 1))
    for k in range(1, n_inst):
        kind = k % 5
        if kind == 1:
            lo[k, 3] = hi[k, 3] = 50 + k                  # settles early
        elif kind == 2:
            hi[k, 1] = 8000                               # fails late
        elif kind == 3:
            lo[k, 4], hi[k, 4] = 3, 2                     # empty
        elif kind == 4:
            hi[k, 1] = 20                                 # fails early
    lo_o, hi_o = lo.reshape(-1).copy(), hi.reshape(-1).copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, threads=8)
    b = pcx.Batch(pir, n_inst, V)
    b.load(lo.reshape(-1), hi.reshape(-1))
    rg, st = b.run(mode)
    lg, ug = b.read()
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(lg.reshape(n_inst, V)[~fo], lo_o.reshape(n_inst, V)[~fo])
    assert np.array_equal(ug.reshape(n_inst, V)[~fo], hi_o.reshape(n_inst, V)[~fo])
    assert rg.sweeps[0] >= 12000 and rg.evals[0] >= 3 * 11999 and rg.has_changed[0]
    assert st.full_launches >= 3                          # 12,000 steps of at most 4,096
    for k in range(1, n_inst):
        if k % 5 == 1:
            assert 50 + k <= rg.sweeps[k] and rg.evals[k] < 12000
        elif k % 5 == 3:
            assert rg.sweeps[k] == 0 and rg.evals[k] == 0
    b.reset()
    lr, ur = b.read()
    assert np.array_equal(lr, lo.reshape(-1)) and np.array_equal(ur, hi.reshape(-1))
