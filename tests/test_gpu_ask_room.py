"""pcx_batch_ask where the caller's room for positions is far above their number: a
safe bound costs neither device memory nor time, and the answers are those of a
call with exactly enough room."""
import ctypes

import numpy as np
import pytest

import pc_ask as pa
import pcx
import pcx.device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


def _sums(P, V, seed):
    """P sums i + j = k over V variables whose solution is their own number."""
    rng = np.random.default_rng(seed)
    y = rng.integers(0, V // 2, P)
    z = rng.integers(0, V // 2, P)
    return np.full(P, pcx.ADD, np.int32), (y + z).astype(np.int32), y.astype(np.int32), z.astype(np.int32)


# 20 M pairs: positions of all of them are above the 64 MB kept; 80,000 M pairs: above
# the device's memory (320 GB).
@pytest.mark.parametrize("n,V,P", [(400, 1000, 50000), (80000, 100, 1000000)])
def test_room_for_every_pair(gpu, n, V, P):
    pir = pcx.PIR()
    pir.tell(*_sums(P, V, n))
    lo = np.tile(np.arange(V, dtype=np.int32), (n, 1))
    hi = lo.copy()
    hi[3, 7] += 1                                        # open in two stores
    hi[n - 1, V // 2] += 2
    b = pcx.Batch(pir, n, V)
    b.load(lo.reshape(-1), hi.reshape(-1))
    ext, off, idx = b.ask()
    assert np.array_equal(np.nonzero(~ext)[0], [3, n - 1]) and 0 < len(idx) < 10 * P
    off2, idx2 = np.zeros(n + 1, np.int64), np.full(len(idx) + 8, -7, np.int32)
    st = pcx.lib().pcx_batch_ask(b._h, None, pcx._p64(off2), pcx._p32(idx2), ctypes.c_int64(n * P))
    assert st == pcx.OK, pcx.lib().pcx_last_error()
    assert np.array_equal(off2, off) and np.array_equal(idx2[:len(idx)], idx) and (idx2[len(idx):] == -7).all()


def _free():
    h = pcx.device._runtime()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert h.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_large_work_arrays_are_given_back(gpu):
    """4,096 stores: 200 MB of answer bits at 400,000 propagators, a 640 MB copy for
    formulas at 20,000 variables.  What a batch keeps between calls stays below 64 MB."""
    n, V, P = 4096, 20000, 400000
    pir = pcx.PIR()
    pir.tell(*_sums(P, V, 1))
    lo = np.tile(np.arange(V, dtype=np.int32), (n, 1)).reshape(-1)
    hi = lo.copy()
    hi[5 * V + 9] += 1
    b = pcx.Batch(pir, n, V)
    b.load(lo, hi)
    b.ask(live=False)                                    # the table goes to the device
    before = _free()
    nodes = np.array([[pa.VAR, 9, 0, 0], [pa.CONST, 9, 0, 0], [pa.EQ, 0, 0, 0]] * 14000, np.int32)
    for _ in range(2):
        ext, _, idx = b.ask()
        assert np.array_equal(np.nonzero(~ext)[0], [5]) and len(idx) > 0
        got = b.ask_formulas(nodes, np.arange(0, 42001, 3, dtype=np.int64))
        assert np.array_equal(np.nonzero(~got)[0], [5])
    assert before - _free() < 96 << 20
    assert np.array_equal(b.read()[1], hi)


@pytest.mark.parametrize("V", [1000, 100000])
def test_few_formulas_copy_no_stores(gpu, V):
    """Below two nodes a variable the stores are not interleaved for an ask (51 MB at
    100,000 variables), and the answers are those of the lanes' kernel from there on."""
    n = 64
    lo = np.tile(np.arange(V, dtype=np.int32), (n, 1))
    hi = lo.copy()
    hi[7, 3] += 1
    lo[9, 5], hi[9, 5] = 4, 2                             # an empty store
    b = pcx.Batch(pcx.PIR(), n, V)
    b.load(lo.reshape(-1), hi.reshape(-1))
    tree = [[pa.VAR, 3, 0, 0], [pa.CONST, 3, 0, 0], [pa.EQ, 0, 0, 0]]
    want = ~np.isin(np.arange(n), (7, 9))

    def ask(m):
        off = np.arange(m + 1, dtype=np.int64) * 3
        return b.ask_formulas(np.array(tree * m, np.int32), off)

    assert np.array_equal(ask(1), want)
    before = _free()
    for m in (1, 50, (2 * V - 1) // 3):                  # up to one node short of the rule
        assert np.array_equal(ask(m), want)
    assert before - _free() < 24 << 20
    for m in ((2 * V + 2) // 3, V):
        assert np.array_equal(ask(m), want)
    lo2, hi2 = b.read()
    assert np.array_equal(lo2, lo.reshape(-1)) and np.array_equal(hi2, hi.reshape(-1))
