"""GPU: the plans of the implicit `A*u` / `mul_` path.  Owners of one structure that live side by
side keep their own values (bitwise equal to fresh plans, no plan made after the first use of
each); an owner that goes leaves its plan to the next one of its structure on that stream; inside
a stream capture, where nothing can be allocated, a live owner's plan may be taken and that owner
still gives its own values afterwards."""
import gc
import threading

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu

N = 91    # a size no other test uses: the pool's plans of this structure are this file's


def owner(g):
    h = 1.0 / (N + 1)
    return D.CenteredDifference(2, 4, h, N) * D.DirichletBC(g, -2 * g)


def field(seed):
    return torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, N)).to("cuda")


def fresh(g, u):
    out = torch.empty_like(u)
    D.plans_for(owner(g), u)[0].apply(out, u)
    return out


@pytest.fixture
def made(monkeypatch):
    import diffeqoperators_amd.apply as ap
    count = []
    orig = ap.Plan.__init__
    monkeypatch.setattr(ap.Plan, "__init__", lambda self, *a, **k: (count.append(1), orig(self, *a, **k))[1])
    return count


def test_live_owners_in_turn_and_reuse(made):
    u = field(1)
    A = [owner(g) for g in (0.5, 1.5, 2.5)]
    want = [fresh(g, u) for g in (0.5, 1.5, 2.5)]
    for a, w in zip(A, want):
        assert torch.equal(a * u, w)
    n = len(made)
    for _ in range(3):
        for a, w in zip(A, want):
            assert torch.equal(a * u, w)
    assert len(made) == n          # no plan made, none rebound to another's values
    du = torch.empty_like(u)
    del A, a
    gc.collect()
    for k in range(20):            # temporaries of the structure reuse a plan that was left
        D.mul_(du, owner(0.1 * k), u)
        assert len(made) == n
        assert torch.equal(du, fresh(0.1 * k, u))
        n = len(made)
    with pytest.raises(TypeError):
        D.mul_(torch.empty(N, dtype=torch.float32, device="cuda"), owner(1.0), u)
    with pytest.raises(ValueError):
        D.mul_(u, owner(1.0), u)


def test_streams_and_threads():
    u = field(2)
    side = torch.cuda.Stream()
    a = owner(3.0)
    want = fresh(3.0, u)
    assert torch.equal(a * u, want)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        got = a * u
    side.synchronize()
    assert torch.equal(got, want)
    del a                          # applied on two streams: its plan is not handed on
    errs = []

    def work(t):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                v = field(10 + t)
                for k in range(20):
                    got = owner(t + 0.01 * k) * v
                    ok = torch.equal(got, fresh(t + 0.01 * k, v))
                    if not ok:
                        errs.append((t, k))
        except Exception as e:     # noqa: BLE001
            errs.append(e)
    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errs


def test_capture_takes_a_live_owners_plan():
    u = field(3)
    a = owner(4.0)
    want = a * u
    out = torch.empty_like(u)
    b = owner(5.0)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        D.mul_(out, b, u)
    for _ in range(3):
        out.zero_()
        g.replay()
        assert torch.equal(out, fresh(5.0, u))
        assert torch.equal(a * u, want)
