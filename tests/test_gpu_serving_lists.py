"""A server's admissions and hand-backs by list (one launch a tick): more requests
in one tick than a list holds (1,024), of which some start from their network's
root fixpoint, some lie outside the told store, some are empty and some fail; every
result equals the request run alone."""
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


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2100])
def test_many_requests_in_one_tick(gpu, n):
    pirs, stores = [], []
    for j, (V, P) in enumerate(((80, 150), (97, 301))):
        op, x, y, z, lb, ub, _ = pcx.gen_network(pcx.gen_params(seed=3 + j, nvars=V, nprops=P, chain_len=10))
        pir = pcx.PIR()
        pir.tell(op, x, y, z, lb, ub)
        pirs.append(pir)
        stores.append((lb, ub))
    srv = pcx.Server(max_slots=2200)
    for j, pir in enumerate(pirs):
        net = srv.add_network(pir)
        if j == 0:
            srv.set_root(net, *stores[0])
    want, work = [], []
    for i in range(n):
        net = i % 2
        lb, ub = stores[net]
        lo, hi = pcx.gen_splits(100 + i, lb, ub, 1, 1, 3)
        if i % 5 == 3:                                   # outside the told store
            v = i % len(lb)
            lo[v], hi[v] = lo[v] - 1, hi[v] + 1
        if i % 11 == 7:
            lo[5], hi[5] = 9, 8                          # empty
        lo_o, hi_o = lo.copy(), hi.copy()
        want.append((lo.copy(), hi.copy(), lo_o, hi_o, ol.fixpoint(*pirs[net].table(), lo_o, hi_o)))
        work.append((lo, hi))
        srv.submit(net, lo, hi, i)
    done = {}
    for _ in range(100000):
        left = srv.step()
        for tag, r, _ in srv.poll(4096):
            done[tag] = (bool(r.failed), bool(r.has_changed))
        if not left:
            break
    assert sorted(done) == list(range(n))
    for i, (lo, hi, lo_o, hi_o, ro) in enumerate(want):
        assert done[i][0] == bool(ro.failed), i
        if not ro.failed:
            assert np.array_equal(work[i][0], lo_o) and np.array_equal(work[i][1], hi_o), i
            assert done[i][1] == bool((lo != lo_o).any() or (hi != hi_o).any()), i
