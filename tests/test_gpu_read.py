"""Batch reads into host memory by several threads (pcx_xfer.hip): sizes around the
threshold, the threads' shares and the slots, whole interval and bitset stores
back as they were loaded; and two engines reading at once, of which one finds the
pool of slots in use."""
import threading

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


def _interval_batch(n, V, seed):
    rng = np.random.default_rng(seed)
    pir = pcx.PIR()
    pir.tell([pcx.ADD], [0], [1], [2])
    lb = rng.integers(-1000, 1000, n * V).astype(np.int32)
    ub = lb + rng.integers(0, 1000, n * V).astype(np.int32)
    b = pcx.Batch(pir, n, V)
    b.load(lb, ub)
    return b, lb, ub


@pytest.mark.parametrize("values", [MB // 8 - 1, MB // 8, MB // 8 + 1, MB // 4 - 3, MB // 4 + 1, MB - 5, MB + 7,
                                    3 * MB + 1])
def test_interval_read(gpu, values):
    b, lb, ub = _interval_batch(1, values, values)
    for _ in range(2):
        lo, hi = b.read()
        assert np.array_equal(lo, lb) and np.array_equal(hi, ub)


@pytest.mark.parametrize("words", [MB // 8 - 1, MB // 8 + 1, MB + 3])
def test_bitset_read(gpu, words):
    rng = np.random.default_rng(words)
    pir = pcx.BitsPIR()
    pir.tell([pcx.BLEQ], [0], [1], [2])
    w = rng.integers(1, 1 << 62, words).astype(np.uint64)
    b = pcx.Batch(pir, 1, words)
    b.load_words(w)
    assert np.array_equal(b.read_words(), w)


def test_two_engines_read_at_once(gpu):
    bs = [_interval_batch(3, 200001, s) for s in (1, 2)]
    bad = []

    def read(b, lb, ub):
        for _ in range(10):
            lo, hi = b.read()
            if not (np.array_equal(lo, lb) and np.array_equal(hi, ub)):
                bad.append(1)

    th = [threading.Thread(target=read, args=x) for x in bs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
