"""Full sweeps of one store whose waves chase what they tighten (pcx_chase.hip),
against the oracle bit for bit: PIR.fixpoint and fixpoint_noalloc with the LDS
kernel off, so that small tables take them too."""
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


def _check(pir, lb, ub, what):
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
    return rg


@pytest.mark.parametrize("P", [63, 64, 65, 255, 256, 257, 5000, 70001, 300007])
def test_networks(gpu, P):
    """Tables around a wave's and a workgroup's 64 and 256 propagators, and some
    of several workgroups per wave's turn; told, empty at the start, failing, and
    the fixpoint again."""
    V = max(80, P // 4 + 1)
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=P, nvars=V, nprops=P, chain_len=50))
    pir = pcx.PIR(lds_mode=0)
    pir.tell(op, x, y, z, lb, ub)
    _check(pir, lb, ub, "told")
    lo, hi = lb.copy(), ub.copy()
    lo[V - 1], hi[V - 1] = 3, 2
    assert _check(pir, lo, hi, "empty at the start").sweeps == 0
    top, tx, ty, tz = pir.table()
    p = int(np.nonzero(np.isin(top, (pcx.ADD, pcx.MIN, pcx.MAX)))[0][-1])
    lo, hi = lb.copy(), ub.copy()
    lo[tx[p]], hi[tx[p]] = hi[tx[p]] + 1000000, hi[tx[p]] + 1000000
    _check(pir, lo, hi, "fails")
    lo, hi = lb.copy(), ub.copy()
    pir.fixpoint(lo, hi)
    assert not _check(pir, lo, hi, "at the fixpoint").has_changed


@pytest.mark.parametrize("fan", [60, 1024, 1100, 6000])
def test_a_late_fan_out(gpu, fan):
    """A chain whose end tightens `fan` propagators at once, each the start of
    another link: more neighbours than the 64 lanes and the 1,024 entries of the
    ring of the wave that chases the chain, which drops the rest for the next
    sweep."""
    L = 300
    x, y = [], []
    for i in range(L):
        x.append(i + 1)
        y.append(i)
    for j in range(fan):
        x += [L + 2 + 2 * j, L + 3 + 2 * j]
        y += [L, L + 2 + 2 * j]
    n = L + 2 + 2 * fan
    lb, ub = np.zeros(n, np.int32), np.full(n, 1000000, np.int32)
    ub[0] = 0
    lb[L + 1] = ub[L + 1] = 1
    pir = pcx.PIR(lds_mode=0)
    pir.tell(np.full(len(x), pcx.ADD), np.array(x), np.array(y), np.full(len(x), L + 1))
    _check(pir, lb, ub, f"fan of {fan}")
    hi = ub.copy()
    hi[n - 1] = L
    assert _check(pir, lb, hi, "fails at the end").failed


@pytest.mark.parametrize("seed", range(6))
def test_random_tables_of_every_opcode(gpu, seed):
    """Random operands (some of them the same variable) and opcodes, divisions
    among them, over small boxes and infinite bounds."""
    rng = np.random.default_rng(seed)
    V, P = 60, 9
    for k in range(16):
        op = rng.integers(0, 10, P)
        x, y, z = rng.integers(0, V, (3, P))
        lb = rng.integers(-20, 5, V).astype(np.int32)
        ub = (lb + rng.integers(0, 2000, V)).astype(np.int32)
        inf = rng.random(V) < 0.2
        lb[inf], ub[inf] = pcx.MINF, pcx.INF
        pir = pcx.PIR(lds_mode=0)
        pir.tell(op, x, y, z, lb, ub)
        if (lb > ub).any():
            continue
        # a table may climb for ever between infinite bounds: bounded for the oracle
        lo, hi = lb.copy(), ub.copy()
        if ol.fixpoint(*pir.table(), lo, hi, max_sweeps=2000).sweeps >= 2000:
            continue
        _check(pir, lb, ub, f"table {seed}.{k}")
