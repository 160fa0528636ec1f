"""Formula asks by a wave's lanes (16 stores or more) and by a thread per store and
formula (fewer): store counts around the groups of 64, formula counts around a
wave's turn of 8 and the check's workgroup of 256, the deepest stack, against the
oracle; malformed trees among many good ones."""
import numpy as np
import pytest

import oracle_lib as ol
import pc_ask as pa
import pcx
from test_gpu_formulas import V, _formula, _stores

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


def _pack(forms):
    nodes = np.array([nd for f in forms for nd in f], np.int32).reshape(-1, 4)
    return nodes, np.cumsum([0] + [len(f) for f in forms]).astype(np.int64)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 130])
def test_store_counts(gpu, n):
    rng = np.random.default_rng(n)
    lo, hi = _stores(rng, n)
    lo[n // 2, 2], hi[n // 2, 2] = 4, 2                   # an empty store
    b = pcx.Batch(pcx.PIR(), n, V)
    b.load(lo.ravel(), hi.ravel())
    for _ in range(12):
        forms = []
        for _ in range(int(rng.integers(1, 4))):
            out = []
            _formula(rng, 3, out)
            forms.append(out)
        nodes, off = _pack(forms)
        want = np.array([pa.is_extractable(nodes, off, lo[k], hi[k], ol.ask) for k in range(n)])
        assert np.array_equal(b.ask_formulas(nodes, off), want)
    lo2, hi2 = b.read()                                    # the ask leaves the stores and the image alone
    assert np.array_equal(lo2, lo.ravel()) and np.array_equal(hi2, hi.ravel())
    b.reset()
    assert np.array_equal(b.read()[0], lo.ravel())


@pytest.mark.parametrize("m", [7, 8, 9, 255, 256, 257, 5000])
def test_formula_counts(gpu, m):
    """Store k has x = k: of m formulas x != j, the one with j = k is not asked,
    wherever it stands."""
    n = 80
    x = np.arange(n, dtype=np.int32) * ((m + 20) // n + 1)
    stores = np.zeros((n, 2), np.int32)
    stores[:, 0] = x
    b = pcx.Batch(pcx.PIR(), n, 2)
    b.load(stores.ravel(), stores.ravel())
    forms = [[(pa.VAR, 0, 0, 0), (pa.CONST, j, 0, 0), (pa.NE, 0, 0, 0)] for j in range(m)]
    assert np.array_equal(b.ask_formulas(*_pack(forms)), x >= m)


def test_the_deepest_stack(gpu):
    """A conjunction of 32 operands, each true in all stores but one."""
    n = 70
    stores = np.zeros((n, 2), np.int32)
    stores[:, 0] = np.arange(n)
    b = pcx.Batch(pcx.PIR(), n, 2)
    b.load(stores.ravel(), stores.ravel())
    one = [(pa.VAR, 0, 0, 0), (pa.LIT, 0, 0, 0)]           # x != 0
    f = one * 32 + [(pa.AND, 32, 0, 0)]
    assert np.array_equal(b.ask_formulas(*_pack([f])), np.arange(n) != 0)


def test_a_malformed_tree_among_good_ones(gpu):
    n = 20
    b = pcx.Batch(pcx.PIR(), n, 4)
    b.load(np.zeros(4 * n, np.int32), np.ones(4 * n, np.int32))
    good = [(pa.VAR, 0, 0, 0), (pa.CONST, 1, 0, 0), (pa.LE, 0, 0, 0)]
    for bad in ([(pa.VAR, 4, 0, 0), (pa.LIT, 0, 0, 0)], [(pa.ADD, 0, 0, 0)], [(pa.AND, -1, 0, 0)],
                [(pa.PROP, 0, 0, 1), (pa.PROP_Z, 9, 0, 0)], []):
        nodes, off = _pack([good] * 300 + [bad] + [good] * 300)
        with pytest.raises(pcx.PcxError) as e:
            b.ask_formulas(nodes, off)
        assert e.value.status == pcx.EINVAL and "formula trees" in str(e.value), bad
    nodes, off = _pack([good] * 10)
    off[4], off[5] = off[5], off[4]                        # offsets that decrease
    with pytest.raises(pcx.PcxError):
        b.ask_formulas(nodes, off)
    assert b.ask_formulas(*_pack([good] * 10)).all()
