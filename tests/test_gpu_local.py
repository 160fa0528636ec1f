"""Fixpoints of stores that fit in a workgroup's LDS (pcx_local.hip): the sizes
where its bitmaps, lists and stacks have edges, against the oracle bit for bit.

The kernel is reached through PIR.fixpoint and fixpoint_noalloc (one store of
separate bounds), Batch.run in persistent mode and, for unseeded interval
batches, in batched mode; batches of more instances than compute units take
narrower workgroups.
"""
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


def _told(net):
    op, x, y, z, lb, ub = (a.copy() for a in net[:6])
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    return pir, lb, ub


def _check_single(pir, lb, ub, what):
    lo, hi = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo, hi)
    lg, ug = lb.copy(), ub.copy()
    rg = pir.fixpoint(lg, ug)
    assert bool(rg.failed) == bool(ro.failed), what
    d_lb, d_ub = DeviceArray(lb), DeviceArray(ub)
    rn = pir.fixpoint_noalloc(d_lb.ptr, d_ub.ptr, len(lb))
    assert bool(rn.failed) == bool(ro.failed), what
    if not ro.failed:
        assert bool(rg.has_changed) == bool(ro.has_changed) == bool(rn.has_changed), what
        assert np.array_equal(lg, lo) and np.array_equal(ug, hi), what
        assert np.array_equal(d_lb.read(), lo) and np.array_equal(d_ub.read(), hi), what
    d_lb.close()
    d_ub.close()


def _check_batch(pir, lo, hi, V, mode, off=None, idx=None):
    n = len(lo) // V
    lo_o, hi_o = lo.copy(), hi.copy()
    ro = ol.fixpoint_batch(*pir.table(), lo_o, hi_o, V, idx=None if idx is None else idx.astype(np.int64), off=off,
                           threads=8)
    b = pcx.Batch(pir, n, V, off, idx)
    b.load(lo, hi)
    rg, st = b.run(mode)
    lg, ug = b.read()
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    ok = ~fo
    for g, o in ((lg, lo_o), (ug, hi_o)):
        assert np.array_equal(g.reshape(n, V)[ok], o.reshape(n, V)[ok])
    assert np.array_equal((rg.has_changed != 0)[ok], np.array([r.has_changed for r in ro], bool)[ok])
    b.reset()
    lr, ur = b.read()
    assert np.array_equal(lr, lo) and np.array_equal(ur, hi), "reset after the run"
    return st, ok


@pytest.mark.parametrize("P", [31, 32, 33, 63, 64, 65, 1000, 2048, 12007, 16384, 16385, 49152])
def test_single_store(gpu, P):
    """Tables around the bitmap's words and the lists' room, up to 16,384
    propagators, the largest that one store takes to this kernel, and beyond; the
    told store, one that starts empty and one that fails."""
    V = max(80, P // 4 + 1)
    net = pcx.gen_network(pcx.gen_params(seed=P, nvars=V, nprops=P, chain_len=50))
    pir, lb, ub = _told(net)
    _check_single(pir, lb, ub, "told")
    lo, hi = lb.copy(), ub.copy()
    lo[V - 1], hi[V - 1] = 3, 2
    _check_single(pir, lo, hi, "empty at the start")
    top, tx, ty, tz = pir.table()
    p = int(np.nonzero(np.isin(top, (pcx.ADD, pcx.MIN, pcx.MAX)))[0][-1])
    lo, hi = lb.copy(), ub.copy()
    lo[tx[p]], hi[tx[p]] = hi[tx[p]] + 1000000, hi[tx[p]] + 1000000
    _check_single(pir, lo, hi, "fails")


def test_one_propagator(gpu):
    pir = pcx.PIR()
    pir.tell([pcx.ADD], [0], [1], [2])
    _check_single(pir, np.array([0, 2, 3], np.int32), np.array([9, 4, 5], np.int32), "one ADD")
    pir = pcx.PIR()
    pir.tell([pcx.ADD], [0], [0], [1])               # x = x + y: its own neighbour
    _check_single(pir, np.array([0, 0], np.int32), np.array([50, 7], np.int32), "x = x + y")


@pytest.mark.parametrize("fan", [100, 129, 5000])
def test_a_late_fan_out(gpu, fan):
    """A chain whose end tightens `fan` propagators at once, each the start of
    another link: the wave that chases the chain finds more marks than its lanes
    and its stack hold (128 entries beside 64 lanes)."""
    L = 300
    n = L + 2 + 2 * fan
    x, y = [], []
    for i in range(L):
        x.append(i + 1)
        y.append(i)
    for j in range(fan):
        x += [L + 2 + 2 * j, L + 3 + 2 * j]
        y += [L, L + 2 + 2 * j]
    P = len(x)
    lb, ub = np.zeros(n, np.int32), np.full(n, 1000000, np.int32)
    ub[0] = 0
    lb[L + 1] = ub[L + 1] = 1
    pir = pcx.PIR()
    pir.tell(np.full(P, pcx.ADD), np.array(x), np.array(y), np.full(P, L + 1))
    _check_single(pir, lb, ub, f"fan of {fan}")
    lo, hi = np.tile(lb, 3), np.tile(ub, 3)
    hi[2 * n + n - 1] = L                            # instance 2 fails at the end of the chain
    st, ok = _check_batch(pir, lo, hi, n, pcx.MODE_PERSISTENT)
    assert list(ok) == [True, True, False]


@pytest.mark.parametrize("n_inst,V,P,mode", [
    (3, 15000, 70001, pcx.MODE_PERSISTENT),          # 32-bit list entries, offsets outside LDS
    (5, 4001, 16003, pcx.MODE_BATCHED),
    (600, 500, 2001, pcx.MODE_BATCHED),              # more instances than compute units
    (600, 500, 2001, pcx.MODE_PERSISTENT),
    (1, 16000, 64001, pcx.MODE_BATCHED),
])
@pytest.mark.parametrize("subsets", [False, True], ids=["whole", "subsets"])
def test_batches(gpu, n_inst, V, P, mode, subsets):
    """Splits of a told store (nothing propagated: no seeded run), with and
    without subsets; one instance starts empty."""
    net = pcx.gen_network(pcx.gen_params(seed=7, nvars=V, nprops=P, chain_len=40))
    pir, lb, ub = _told(net)
    lo, hi = pcx.gen_splits(8, lb, ub, n_inst, 1, 4)
    if n_inst > 2:
        lo[2 * V + 1], hi[2 * V + 1] = 5, 4
    off, idx = pcx.gen_subsets(9, P, n_inst, P // 10, P) if subsets else (None, None)
    st, ok = _check_batch(pir, lo, hi, V, mode, off, idx)
    sizes = np.full(n_inst, P) if off is None else np.diff(off)
    assert st.full_launches == 1 and st.full_evals == int(sizes.sum()) - (int(sizes[2]) if n_inst > 2 else 0)


@pytest.mark.parametrize("n_inst", [4, 300])
def test_bitset_batches(gpu, n_inst):
    """Bitset stores in persistent mode."""
    V, P = 700, 2801
    op, x, y, z, words = pcx.gen_bits_network(5, V, P)
    pir = pcx.BitsPIR()
    pir.tell(op, x, y, z, words)
    w = pcx.gen_bits_splits(6, words, n_inst, 1, 6)
    wo = w.copy()
    ro = ol.bits_fixpoint_batch(*pir.table(), wo, V, threads=8)
    b = pcx.Batch(pir, n_inst, V)
    b.load_words(w)
    rg, st = b.run(pcx.MODE_PERSISTENT)
    fo = np.array([r.failed for r in ro], bool)
    assert np.array_equal(rg.failed != 0, fo)
    assert np.array_equal(b.read_words().reshape(n_inst, V)[~fo], wo.reshape(n_inst, V)[~fo])
