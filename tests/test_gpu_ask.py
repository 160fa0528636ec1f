"""pcx_batch_ask around its chunks of 4,096 propagators and words of 64: open
propagators and extractability against PIR.ask_all on each store; stores that just
fit in a workgroup's LDS (160 KB) and that do not."""
import ctypes

import numpy as np
import pytest

import pcx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    if pcx.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return True


def _case(n, V, P, seed):
    op, x, y, z, lb, ub, w = pcx.gen_network(pcx.gen_params(seed=seed, nvars=V, nprops=P, chain_len=20))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    pir.fixpoint(lb, ub)
    lo, hi = pcx.gen_splits(seed + 1, lb, ub, n, 0, 3)
    lo, hi = lo.reshape(n, V), hi.reshape(n, V)
    lo[0], hi[0] = w, w                                  # the solution: nothing is open
    if n > 2:
        lo[2, V - 1], hi[2, V - 1] = 5, 4                # an empty store
    return pir, lo, hi


@pytest.mark.parametrize("n,V,P", [(1, 80, 63), (3, 80, 64), (3, 80, 65), (4, 1100, 4095), (4, 1100, 4096),
                                   (4, 1100, 4097), (3, 2100, 8193), (300, 120, 400),
                                   (3, 20400, 9000), (3, 20500, 9000)])
@pytest.mark.parametrize("subsets", [False, True], ids=["whole", "subsets"])
def test_ask(gpu, n, V, P, subsets):
    pir, lo, hi = _case(n, V, P, P)
    off = idx = None
    if subsets:
        off, idx = pcx.gen_subsets(3, P, n, 0, P)
        if n > 1:                                        # instance 1 has no propagator
            idx = np.concatenate([idx[:off[1]], idx[off[2]:]])
            off = np.concatenate([off[:2], off[2:] - (off[2] - off[1])])
    b = pcx.Batch(pir, n, V, off, idx)
    b.load(lo.reshape(-1), hi.reshape(-1))
    ext, loff, lidx = b.ask()
    for k in range(n):
        ent, _ = pir.ask_all(lo[k].copy(), hi[k].copy())
        mine = np.arange(P) if off is None else idx[off[k]:off[k + 1]]
        want = mine[~ent[mine]]
        assert np.array_equal(lidx[loff[k]:loff[k + 1]], want), k
        assert ext[k] == (len(want) == 0 and not (lo[k] > hi[k]).any()), k
    assert ext[0]
    ext2, none, _ = b.ask(live=False)
    assert np.array_equal(ext2, ext) and none is None
    # too little room: refused, with the size needed; nothing is written
    total = int(loff[-1])
    if total:
        got, few = np.zeros(n + 1, np.int64), np.full(total, -7, np.int32)
        st = pcx.lib().pcx_batch_ask(b._h, None, pcx._p64(got), pcx._p32(few), ctypes.c_int64(total - 1))
        assert st == pcx.EINVAL and got[-1] == total and (few == -7).all()
