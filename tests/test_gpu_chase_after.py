"""Stores chased after the plain sweeps that a table of their size gets first
(pcx_internal.h: eight up to 1,048,576 propagators, four beyond), against the
oracle: tables of both sides of that line, and chains of every opcode that are
longer than the plain sweeps reach."""
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


def _check(pir, lb, ub):
    lo, hi = lb.copy(), ub.copy()
    ro = ol.fixpoint(*pir.table(), lo, hi)
    lg, ug = lb.copy(), ub.copy()
    rg = pir.fixpoint(lg, ug)
    d_lb, d_ub = DeviceArray(lb), DeviceArray(ub)
    rn = pir.fixpoint_noalloc(d_lb.ptr, d_ub.ptr, len(lb))
    assert bool(rg.failed) == bool(rn.failed) == bool(ro.failed)
    if not ro.failed:
        assert bool(rg.has_changed) == bool(rn.has_changed) == bool(ro.has_changed)
        assert np.array_equal(lg, lo) and np.array_equal(ug, hi)
        assert np.array_equal(d_lb.read(), lo) and np.array_equal(d_ub.read(), hi)
    d_lb.close()
    d_ub.close()
    return rg


@pytest.mark.parametrize("P", [(1 << 20) - 1, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("links", [3, 6, 40])
def test_tables_at_the_line(gpu, P, links):
    op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=links, nvars=P // 4, nprops=P, chain_len=links))
    pir = pcx.PIR()
    pir.tell(op, x, y, z, lb, ub)
    assert pir.table()[0].size == P
    assert _check(pir, lb, ub).has_changed


@pytest.mark.parametrize("links", [8, 12, 200])
@pytest.mark.parametrize("seed", range(4))
def test_chains_of_every_opcode(gpu, seed, links):
    """400 chains whose first variable is told: each link one random opcode on the
    variable before and a constant, shuffled over the table."""
    rng = np.random.default_rng(seed * 1000 + links)
    n = 400
    v = np.arange(n * (links + 1)).reshape(n, links + 1)
    consts = v.size + np.arange(6)
    V = v.size + 6
    lb, ub = np.full(V, -100000, np.int32), np.full(V, 100000, np.int32)
    ub[v[:, 0]] = rng.integers(-50, 50, n)
    lb[v[:, 0]] = ub[v[:, 0]] - rng.integers(0, 20, n)
    lb[consts] = ub[consts] = [-1, 1, -3, 2, 5, 7]
    x, y = v[:, 1:].reshape(-1), v[:, :-1].reshape(-1)
    p = rng.permutation(x.size)
    op = rng.choice([ol.OPS["ADD"], ol.OPS["ADD"], ol.OPS["MIN"], ol.OPS["MAX"]] + list(range(10)), x.size)
    z = np.where(op == ol.OPS["MUL"], rng.choice(consts[:2], x.size), rng.choice(consts, x.size))
    pir = pcx.PIR(lds_mode=0)
    pir.tell(op.astype(np.int32), x[p].astype(np.int32), y[p].astype(np.int32), z.astype(np.int32), lb, ub)
    _check(pir, lb, ub)
