"""Large reads before and after a program's reads are worth the pinned slots (32 MB of
them with an engine alive): the same results from both ways, around the megabyte from
which the slots are used and the ends of their shares."""
import numpy as np
import pytest

import pcx

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


def _batch(values, seed):
    rng = np.random.default_rng(seed)
    pir = pcx.PIR()
    pir.tell([pcx.ADD], [0], [1], [2])
    lb = rng.integers(-1000, 1000, values).astype(np.int32)
    ub = lb + rng.integers(0, 1000, values).astype(np.int32)
    b = pcx.Batch(pir, 1, values)
    b.load(lb, ub)
    return b, lb, ub


def _read(b, lb, ub):
    lo, hi = b.read()
    assert np.array_equal(lo, lb) and np.array_equal(hi, ub)


def test_reads_before_and_with_slots(gpu):
    big = _batch(MB, 1)                                   # 8 MB a read
    for _ in range(6):                                    # the slots come with the fifth
        _read(*big)
    for values in (MB // 8 - 1, MB // 8, MB // 8 + 1, MB // 4 - 3, MB // 4 + 1, MB // 2 + 511, MB - 5, MB + 7,
                   3 * MB + 1):
        _read(*_batch(values, values))
    rng = np.random.default_rng(5)
    for words in (MB // 8 - 1, MB // 8 + 1, MB + 3):
        pir = pcx.BitsPIR()
        pir.tell([pcx.BLEQ], [0], [1], [2])
        w = rng.integers(1, 1 << 62, words).astype(np.uint64)
        b = pcx.Batch(pir, 1, words)
        b.load_words(w)
        assert np.array_equal(b.read_words(), w)
    _read(*big)
