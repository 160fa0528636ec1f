"""Children of a branching whose run drains their marks: their image is the drain's undo
log, or a row written when the log is about to overflow.  Runs and resets give the
oracle's stores and the children again, whatever kind of run comes in between."""
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


# links, leaves: a chain from variable 0 (one round a link; past 1,024 tightened variables the
# log overflows) and a star on it (rounds whose propagators alone could fill the log)
SHAPES = {"few": (20, 5), "edge": (1023, 0), "over": (1024, 0), "long": (1500, 7), "dense": (3, 341),
          "wide": (3, 342), "lists": (5, 1500)}


def _net(bits, links, leaves):
    V = 1 + links + leaves + 2                   # variable 0, the chain, the leaves, 0 and a free one
    zero = V - 2
    x = np.arange(1, 1 + links + leaves, dtype=np.int32)
    y = np.concatenate([np.arange(links), np.zeros(leaves)]).astype(np.int32)
    z = np.full(len(x), zero, np.int32)
    if bits:
        w = np.full(V, ol.word(range(6)), np.uint64)
        w[zero] = ol.word([0])
        pir = pcx.BitsPIR()
        pir.tell(np.full(len(x), ol.BITS_OPS["ADD"], np.int32), x, y, z, w)
        return pir, V, w
    lo, hi = np.zeros(V, np.int32), np.full(V, 9, np.int32)
    hi[zero] = 0
    pir = pcx.PIR()
    pir.tell(np.full(len(x), ol.OPS["ADD"], np.int32), x, y, z, lo, hi)
    return pir, V, (lo, hi)


def _read(bits, b):
    return [b.read_words()] if bits else list(b.read())


def _oracle(bits, pir, stores, V):
    t = pir.table()
    out = [s.copy() for s in stores]
    if bits:
        return out, ol.bits_fixpoint_batch(*t, out[0], V)
    return out, ol.fixpoint_batch(*t, out[0], out[1], V)


def _same(got, want):
    return all((g == w).all() for g, w in zip(got, want))


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("bits", [False, True], ids=["intervals", "bits"])
def test_children_keep_their_image(gpu, bits, shape):
    links, leaves = SHAPES[shape]
    pir, V, root = _net(bits, links, leaves)
    n = 3
    parent = pcx.Batch(pir, n, V)
    if bits:
        w = np.tile(root, n)
        w[V + V - 1] = np.uint64(0)              # parent 1 is empty
        parent.load_words(w)
    else:
        lo, hi = np.tile(root[0], n), np.tile(root[1], n)
        hi[2 * V] = 3                            # parent 2 has less to split
        lo[V + V - 1], hi[V + V - 1] = 4, 3      # parent 1 is empty
        parent.load(lo, hi)
    parent.run(pcx.MODE_BATCHED)
    child = pcx.Batch(pir, 2 * n, V)
    grand = pcx.Batch(pir, 4 * n, V)

    def branched():
        parent.branch(child, from_fixpoint=True)
        return _read(bits, child)

    children = branched()
    want, res = _oracle(bits, pir, children, V)
    failed = [r.failed for r in res]

    def ran(mode):
        rg, _ = child.run(mode)
        assert [r.failed for r in rg] == failed
        got = _read(bits, child)
        for k in range(2 * n):
            if not failed[k]:
                assert _same([g[k * V:(k + 1) * V] for g in got], [s[k * V:(k + 1) * V] for s in want])

    for _ in range(2):                           # the second branching finds the planes as a drain left them
        ran(pcx.MODE_BATCHED)
        child.reset()
        assert _same(_read(bits, child), children)
        ran(pcx.MODE_BATCHED)                    # no marks are left: an ordinary run from the image
        child.reset()
        assert _same(_read(bits, child), children)
        assert _same(branched(), children)
    ran(pcx.MODE_PLAIN)                          # never drained
    child.reset()
    assert _same(_read(bits, child), children)
    branched()
    ran(pcx.MODE_BATCHED)
    ran(pcx.MODE_PERSISTENT)                     # from the drained stores, no reset between
    child.reset()
    assert _same(_read(bits, child), children)
    branched()
    pir.set_config(max_sweeps=1)                 # a limit set after the branching: sweeps, no drain
    child.run(pcx.MODE_BATCHED)
    pir.set_config(max_sweeps=0)
    child.reset()
    assert _same(_read(bits, child), children)
    branched()
    ran(pcx.MODE_BATCHED)
    child.branch(grand, from_fixpoint=True)      # a child that branches keeps its own image
    below = _read(bits, grand)
    gw, gres = _oracle(bits, pir, below, V)
    rg, _ = grand.run(pcx.MODE_BATCHED)
    assert [r.failed for r in rg] == [r.failed for r in gres]
    grand.reset()
    assert _same(_read(bits, grand), below)
    child.reset()
    assert _same(_read(bits, child), children)


@pytest.mark.parametrize("n", [3, 1020, 1050], ids=["few", "wide", "narrow"])
@pytest.mark.parametrize("fan", [1, 2, 3, 7, 31, 64, 65, 130, 300])
def test_rounds_of_any_width(gpu, n, fan):
    """A drained round that tightens `fan` variables at once, whose adjacency lists groups of
    64 threads down to one walk (and, past 256 variables, the evaluating threads), one variable
    of them a hub with more propagators than a group has threads; workgroups of both widths."""
    hub = 90
    V = 1 + fan + fan + hub + 1
    zero = V - 1
    x = np.concatenate([1 + np.arange(fan), 1 + fan + np.arange(fan), 1 + 2 * fan + np.arange(hub)]).astype(np.int32)
    y = np.concatenate([np.zeros(fan), 1 + np.arange(fan), np.full(hub, 1)]).astype(np.int32)
    z = np.full(len(x), zero, np.int32)
    lo, hi = np.zeros(V, np.int32), np.full(V, 9, np.int32)
    hi[zero] = 0
    pir = pcx.PIR()
    pir.tell(np.full(len(x), ol.OPS["ADD"], np.int32), x, y, z, lo, hi)
    lb, ub = np.tile(lo, (n, 1)), np.tile(hi, (n, 1))
    lb[:, 0] = np.random.default_rng(fan).integers(0, 9, n)
    parent = pcx.Batch(pir, n, V)
    parent.load(lb.reshape(-1), ub.reshape(-1))
    parent.run(pcx.MODE_BATCHED)
    child = pcx.Batch(pir, 2 * n, V)
    parent.branch(child, from_fixpoint=True)
    ref = [a.copy() for a in child.read()]
    rg, st = child.run(pcx.MODE_BATCHED)
    assert st.full_evals == 0                    # drained
    ro = ol.fixpoint_batch(*pir.table(), ref[0], ref[1], V)
    assert [r.failed for r in rg] == [r.failed for r in ro]
    assert _same(list(child.read()), ref)


@pytest.mark.parametrize("ran", [False, True], ids=["branched", "drained"])
@pytest.mark.parametrize("gi", [0, 16])
def test_children_are_loaded_over(gpu, gi, ran):
    """Stores loaded from device memory into children that hold no image are the new image."""
    from pcx.device import DeviceArray
    pir, V, (lo, hi) = _net(False, 1100, 7)
    pir.set_config(lockstep=gi)
    n = 3
    parent, child = pcx.Batch(pir, n, V), pcx.Batch(pir, 2 * n, V)
    parent.load(np.tile(lo, n), np.tile(hi, n))
    parent.run(pcx.MODE_BATCHED)
    lb, ub = np.tile(lo, 2 * n), np.tile(hi, 2 * n)
    lb[V], ub[4 * V] = 2, 5
    want, res = _oracle(False, pir, [lb, ub], V)
    dev = [DeviceArray(lb), DeviceArray(ub)]
    for _ in range(2):                           # (the second load finds its lists there)
        parent.branch(child, from_fixpoint=True)
        if ran:
            child.run(pcx.MODE_BATCHED)
        child.load_device(dev[0].ptr, dev[1].ptr)
        rg, _ = child.run(pcx.MODE_BATCHED)
        assert [r.failed for r in rg] == [r.failed for r in res]
        assert _same(list(child.read()), want)
        child.reset()
        assert _same(list(child.read()), [lb, ub])
