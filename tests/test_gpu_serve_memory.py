"""GPU: what a server holds of the device's memory.  Its budget bounds the resident requests' state;
the memory itself is taken as requests come (a whole budget per server cost small bursts more
than their steps), and results do not depend on the pieces it is taken in."""
import threading
import time

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu


def request(n, seed, dtype=torch.float32):
    rng = np.random.default_rng(seed)
    h = 1.0 / (n + 1)
    A = (D.CenteredDifference[1](2, 4, h, n) + D.CenteredDifference[2](2, 4, h, n)) * \
        D.compose(*D.Dirichlet0BC(float, (n, n)))
    u0 = torch.from_numpy(rng.uniform(-1, 1, (n, n))).to(dtype).pin_memory()
    return D.plan_for_shape(A, (n, n), dtype), u0, 0.05 * h * h


def serve(srv, reqs, nsteps=3):
    ids = [srv.submit(p, u0, 1.0, dt, nsteps, 0.0) for p, u0, dt in reqs]
    srv.run()
    return [srv.results[i].clone() for i in ids]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_burst_takes_what_it_needs(dtype):
    reqs = [request(n, n, dtype) for n in (64, 90, 131)]
    want = serve(D.Server(1 << 28), reqs)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    srv = D.Server(8 << 30)
    for got, w in zip(serve(srv, reqs), want):
        assert torch.equal(got, w)
    assert before - torch.cuda.mem_get_info()[0] < 256 << 20   # not the 8 GiB


def test_budget_that_is_not_there_is_refused():
    with pytest.raises(D._abi.DopError) as e:
        D.Server(1 << 50)
    assert e.value.code == D._abi.ENOMEM


def test_pieces_and_the_whole_budget():
    # small live requests leave the arena in pieces; one that needs the whole budget then runs too
    n = 512
    big = request(n, 1)
    budget = 4 * n * n * 4
    small = [request(m, m) for m in (64, 70, 101, 130, 64, 90, 180, 64)]
    want = [serve(D.Server(budget), [r])[0] for r in small + [big]]
    srv = D.Server(budget, max_active=4)
    srv.open()
    th = threading.Thread(target=srv.run)
    th.start()
    ids = []
    try:
        for p, u0, dt in small + [big]:
            ids.append(srv.submit(p, u0, 1.0, dt, 3))
            time.sleep(0.002)
    finally:
        srv.close()
        th.join(timeout=60)
    assert not th.is_alive()
    for i, w in zip(ids, want):
        assert torch.equal(srv.results[i], w)
    assert srv.stats()["peak_bytes"] == budget


def test_budgets_of_two_servers_must_fit_together():
    free = torch.cuda.mem_get_info()[0]
    a = D.Server(free * 6 // 10)
    with pytest.raises(D._abi.DopError) as e:
        D.Server(free * 6 // 10)
    assert e.value.code == D._abi.ENOMEM
    p, u0, dt = request(64, 1)
    got = serve(a, [(p, u0, dt)])
    with pytest.raises(D._abi.DopError):
        D.Server(free * 6 // 10)
    del a
    assert torch.equal(got[0], serve(D.Server(free * 6 // 10), [(p, u0, dt)])[0])


def test_a_request_is_resident_until_its_state_is_back():
    # one slot: the second request takes it over while the first one's state (34 MB) is on its way back
    big, small = request(2048, 1, torch.float64), request(64, 2, torch.float64)
    srv = D.Server(1 << 30, max_active=1)
    serve(srv, [big, small], nsteps=1)
    assert srv.stats()["peak_active"] == 1
    srv = D.Server(1 << 30, max_active=2)
    serve(srv, [big, small], nsteps=1)
    assert srv.stats()["peak_active"] == 2
