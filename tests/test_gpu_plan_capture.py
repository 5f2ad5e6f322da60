"""GPU: implicit applies (`A*u`, `mul_`) inside captured graphs.  A graph keeps its plans, with the
values they had: whatever is captured, applied or let go afterwards, every replay gives the values of
the operator that was captured, and eager applies give their own; the plans are given back with
the graph."""
import gc

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu

N = 83    # a size no other test uses


def owner(g, n=N):
    h = 1.0 / (n + 1)
    return D.CenteredDifference(2, 4, h, n) * D.DirichletBC(g, -2 * g)


def field(seed, n=N):
    return torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, n)).to("cuda")


def fresh(g, u):
    out = torch.empty_like(u)
    D.plans_for(owner(g, u.numel()), u)[0].apply(out, u)
    return out


def captured(f):
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        f()
    return g


def test_two_graphs_and_eager_applies_keep_their_values():
    u = field(1)
    a, b = owner(4.0), owner(5.0)
    want = {g: fresh(g, u) for g in (4.0, 5.0)}
    assert torch.equal(a * u, want[4.0])
    oa, ob = torch.empty_like(u), torch.empty_like(u)
    ga = captured(lambda: D.mul_(oa, a, u))
    gb = captured(lambda: D.mul_(ob, b, u))        # never applied before
    assert torch.equal(b * u, want[5.0])           # before any replay
    for _ in range(3):
        for g, o, w in ((gb, ob, 5.0), (ga, oa, 4.0)):
            o.zero_()
            g.replay()
            assert torch.equal(o, want[w])
        assert torch.equal(a * u, want[4.0])
        assert torch.equal(b * u, want[5.0])


def test_owners_that_go_and_pooled_plans():
    u, out = field(2), torch.empty(N, dtype=torch.float64, device="cuda")
    D.mul_(out, owner(1.0), u)                     # leaves a plan to the pool
    first = captured(lambda: D.mul_(out, owner(6.0), u))
    rebound = owner(7.0)
    assert torch.equal(rebound * u, fresh(7.0, u))   # (a pooled plan, updated)
    out2 = torch.empty_like(u)
    second = captured(lambda: D.mul_(out2, rebound, u))
    del rebound
    gc.collect()
    for k in range(20):                            # others of the structure come and go
        w = fresh(0.1 * k, u)
        assert torch.equal(owner(0.1 * k) * u, w)
        out.zero_(), out2.zero_()
        first.replay(), second.replay()
        assert torch.equal(out, fresh(6.0, u))
        assert torch.equal(out2, fresh(7.0, u))


def test_several_streams_and_graphs_of_one_owner():
    u = field(3)
    a = owner(8.0)
    want = fresh(8.0, u)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):                  # the usual warm-up on a side stream
        got = a * u
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    outs = [torch.empty_like(u) for _ in range(3)]
    graphs = []
    for o in outs:
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            for _ in range(2):
                D.mul_(o, a, u)
        graphs.append(g)
    assert torch.equal(a * u, want)
    del a
    gc.collect()
    del graphs[0]
    for k in range(70):                            # more than the pool holds
        owner(k + 0.5) * u
    torch.cuda.synchronize()
    for g, o in zip(graphs, outs[1:]):
        o.zero_()
        g.replay()
        assert torch.equal(o, want)


def test_plans_are_given_back_with_the_graph():
    n = 1 << 20
    u, out = field(4, n), torch.empty(n, dtype=torch.float64, device="cuda")
    dx = (1.0 + 0.1 * np.random.default_rng(5).random(n + 1)) / n   # 25 MB of weights and more

    def temporary():
        return D.CenteredDifference(2, 2, dx, n) * D.DirichletBC(0.0, 1.0)
    want = temporary() * u

    def cycle():
        g = captured(lambda: D.mul_(out, temporary(), u))
        out.zero_()
        g.replay()
        assert torch.equal(out, want)
        g.reset()
        del g
        gc.collect()
        fresh(0.25, field(6))    # (the next plan made frees what graphs have left)
    cycle()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(6):
        cycle()
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 32 << 20


def test_plans_freed_in_a_capture():
    # plans of owners that go while a stream is being captured, and plans that earlier graphs have
    # left: freeing them neither ends the capture nor becomes part of it
    u, out = field(7), torch.empty(N, dtype=torch.float64, device="cuda")
    for k in range(4):
        held = [D.plans_for(owner(0.3 + i), u) for i in range(3)]
        a = owner(9.0 + k)
        gone = captured(lambda: D.mul_(out, owner(0.7), u))

        def work():
            gone.reset()
            held.clear()
            gc.collect()
            D.mul_(out, a, u)
        g = captured(work)
        for _ in range(3):
            out.zero_()
            g.replay()
            assert torch.equal(out, fresh(9.0 + k, u))
