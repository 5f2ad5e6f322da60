"""GPU: one operator applied on several streams (`A*u`, `mul_`).  Its plan may come from the pool, its
values set on the stream that bound it: an apply on another stream waits for them, whoever got the
plan first."""
import gc
import threading

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
import diffeqoperators_amd.apply as ap

pytestmark = pytest.mark.gpu

N = 87    # a size no other test uses


def owner(g):
    h = 1.0 / (N + 1)
    return D.CenteredDifference(2, 4, h, N) * D.DirichletBC(g, -2 * g)


def field(seed):
    return torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, N)).to("cuda")


def fresh(g, u):
    out = torch.empty_like(u)
    D.plans_for(owner(g), u)[0].apply(out, u)
    return out


def pooled():
    return [e for e in list(ap._POOL) if e[0][0] == (N,)]


def test_other_streams_wait_for_a_pooled_plans_values():
    u, want = field(1), fresh(9.0, field(1))
    s1, s2, s3 = (torch.cuda.Stream() for _ in range(3))
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        owner(1.0) * u                              # leaves its plan to the pool, for s1
    torch.cuda.synchronize()
    gc.collect()
    assert len(pooled()) == 1
    outs = []
    with torch.cuda.stream(s1):
        torch.cuda._sleep(20_000_000)
        a = owner(9.0)
        outs.append(a * u)                          # behind the sleep
    assert len(pooled()) == 0
    for s in (s2, s3, s2):
        with torch.cuda.stream(s):
            outs.append(a * u)
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, want)


def test_plans_bound_by_two_threads_at_once_are_not_handed_on():
    u, want = field(2), fresh(3.0, field(2))
    a = owner(3.0)
    outs, streams = [None, None], [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()

    def work(t):
        with torch.cuda.stream(streams[t]):
            outs[t] = a * u

    ts = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    with ap._POOL_LOCK:                             # both find no plan, and wait
        [t.start() for t in ts]
        [t.join(timeout=0.5) for t in ts]
    [t.join() for t in ts]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], want) and torch.equal(outs[1], want)
    before = len(pooled())
    del a, work, ts
    gc.collect()
    assert len(pooled()) == before
