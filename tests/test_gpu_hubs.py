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


@pytest.mark.parametrize("net", NETS)
@pytest.mark.parametrize("F", [0, 60, 93, 94, 95, 96, 97, 98, 99, 100, 2000, 15000])
def test_single_stores_in_lds(gpu, net, F):
    """The LDS kernel: the hub's degree at, below and above 96 + n / 32 and far above;
    and as a batch of one, whose counts go on when sweeps take the store over."""
    tell, lb, ub = NETS[net](60, F)
    pir = _told(tell, lb, ub, F)
    r = _check(pir, lb, ub)
    assert r.sweeps > 1 and r.evals >= len(tell)
    hi = ub.copy()
    hi[1] = 40
    assert _check(pir, lb, hi).failed
    lo_o, hi_o = lb.copy(), ub.copy()
    ol.fixpoint(*pir.table(), lo_o, hi_o)
    for mode in (pcx.MODE_PLAIN, pcx.MODE_BATCHED, pcx.MODE_PERSISTENT):
        b = pcx.Batch(pir, 1, len(lb))
        b.load(lb, ub)
        res, st = b.run(mode)
        l, u = b.read()
        assert not res.failed[0] and res.has_changed[0] and np.array_equal(l, lo_o) and np.array_equal(u, hi_o)
        assert st.evals == res.evals[0] >= len(tell) and st.sweeps_max == res.sweeps[0] > 1
        assert st.tightened >= int((lb != lo_o).sum() + (ub != hi_o).sum())


def _chunky(F):
    """tasks, then two chains off the last task, so that chases with single marks
    follow rounds in which the hub was tightened, and the other way round."""
    tell, lb, ub = _tasks(70, F)
    s, n = 2, len(lb)
    L = 150
    for c in range(2):
        at = n + c * L
        tell += [(pcx.ADD, at, s + 70, 0)] + [(pcx.ADD, at + i + 1, at + i, 0) for i in range(L - 1)]
        tell += [(pcx.LEQ, 0, at + i, 1) for i in range(40 * c, L, 50)]
    lb, ub = np.append(lb, np.zeros(2 * L, np.int32)), np.append(ub, np.full(2 * L, 100000, np.int32))
    return tell, lb.astype(np.int32), ub.astype(np.int32)


@pytest.mark.parametrize("n_inst,mode", [(3, pcx.MODE_PERSISTENT), (9, pcx.MODE_BATCHED),
                                         (600, pcx.MODE_PERSISTENT), (600, pcx.MODE_BATCHED)])
@pytest.mark.parametrize("F", [20, 700, 6000])
@pytest.mark.parametrize("subsets", [False, True], ids=["whole", "subsets"])
def test_batches_in_lds(gpu, n_inst, mode, F, subsets):
    """Instances that settle, fail by a low makespan (in a sweep, a round or a
    chase) or are settled as loaded, with and without subsets."""
    tell, lb, ub = _chunky(F)
    V, P = len(lb), len(tell)
    pir = _told(tell, lb, ub, F, base_seed=0)
    lo, hi = np.tile(lb, (n_inst, 1)), np.tile(ub, (n_inst, 1))
    for k in range(n_inst):
        lo[k, 2] = 5 + k % 7                              # the first task's start
        if k % 3 == 1:
            hi[k, 1] = 30 + 11 * (k % 23)
    rl, ru = lb.copy(), ub.copy()
    ol.fixpoint(*pir.table(), rl, ru)
    lo[2::9], hi[2::9] = rl, ru
    off, idx = pcx.gen_subsets(9, P, n_inst, P // 2, P) if subsets else (None, None)
    lo_o, hi_o = lo.reshape(-1).copy(), hi.reshape(-1).copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, idx=idx.astype(np.int64) if subsets else None, off=off,
                           threads=8)
    b = pcx.Batch(pir, n_inst, V, off, idx)
    b.load(lo.reshape(-1), hi.reshape(-1))
    rg, _ = b.run(mode)
    lg, ug = b.read()
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(lg.reshape(n_inst, V)[~fo], lo_o.reshape(n_inst, V)[~fo])
    assert np.array_equal(ug.reshape(n_inst, V)[~fo], hi_o.reshape(n_inst, V)[~fo])
    assert np.array_equal((rg.has_changed != 0)[~fo], np.array([r.has_changed for r in ro], bool)[~fo])
    assert (rg.sweeps >= 1).all() and (rg.evals >= 1).all()


@pytest.mark.parametrize("n_inst", [3, 300])
def test_bitset_batches_in_lds(gpu, n_inst):
    """Bitset stores in persistent mode: a chain of 50 sums below a hub that 400
    others are below too; every link removes a value of the hub."""
    L, F = 50, 400
    s, o = 2, 3 + L
    tell = [(pcx.BADD, s + i + 1, s + i, 0) for i in range(L)]
    tell += [(pcx.BLEQ, s + i, s + i, 1) for i in range(L + 1)]
    tell += [(pcx.BLEQ, o + j, o + j, 1) for j in range(F)]
    V = 3 + L + F
    words = np.full(V, 2**64 - 1, np.uint64)
    words[0] = 2
    perm = np.random.default_rng(3).permutation(len(tell))
    pir = pcx.BitsPIR()
    pir.tell(*(np.array([p[i] for p in tell], np.int32)[perm] for i in range(4)), words)
    w = np.tile(words, (n_inst, 1))
    for k in range(n_inst):
        w[k, s] = 1 << (k % 12)
        if k % 4 == 3:
            w[k, 1] = (1 << 30) - 1
    w = w.reshape(-1)
    wo = w.copy()
    ro = ol.bits_fixpoint_batch(*pir.table(), wo, V, threads=8)
    b = pcx.Batch(pir, n_inst, V)
    b.load_words(w)
    rg, _ = b.run(pcx.MODE_PERSISTENT)
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(b.read_words().reshape(n_inst, V)[~fo], wo.reshape(n_inst, V)[~fo])
