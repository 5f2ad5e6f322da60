"""GPU: RK4 steps of problems that go stage by stage (periodic BCs, three ghost taps: what the one-pass
steps do not take) in one batch, or one server's size class, with problems that take the one-pass
steps: 1-D and 2-D tiles of every window in one launch a stage, beside the passes.  Against plans of the
generic kernel, whose steps run every stage over the whole grid: bit for bit, after odd and even
numbers of steps."""
import os

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu

# (sizes, derivative, approximation order, BC): windows of 3, 5, 7, 9 and 11 points
CASES = [((n,), d, a, bc) for n, d, a in ((300, 2, 2), (1031, 2, 4), (777, 2, 6), (640, 2, 8), (901, 4, 8))
         for bc in ("periodic", "robin3")]
CASES += [(s, d, a, bc) for s, d, a in (((70, 96), 2, 2), ((131, 140), 2, 4), ((170, 133), 2, 6),
                                        ((150, 211), 2, 8), ((120, 180), 4, 8))
          for bc in ("periodic", "robin3")]
# these take the one-pass steps
CASES += [((1500,), 2, 4, "dirichlet"), ((140, 150), 2, 4, "dirichlet"), ((260, 301), 2, 6, "robin"),
          ((72, 65), 2, 2, "dirichlet"), ((230, 190), 2, 8, "robin")]


def operator(case):
    shape, d, a, bc = case
    js = tuple(reversed(shape))
    A = None
    for N, n in enumerate(js, 1):
        L = D.CenteredDifference[N](d, a, 1.0 / (n + 1), n)
        A = L if A is None else A + L

    def atom(n):
        h = 1.0 / (n + 1)
        if bc == "periodic":
            return D.PeriodicBC(float)
        if bc == "dirichlet":
            return D.DirichletBC(0.2, -0.3)
        return D.RobinBC((1.0, 0.5, 0.1), (1.0, 0.5, -0.2), h, 3 if bc == "robin3" else 1)
    if len(js) == 1:
        return A * atom(js[0])
    return A * D.compose(*(D.MultiDimBC[N](atom(n), js) for N, n in enumerate(js, 1)))


def generic(make):
    os.environ["DOP_FORCE_GENERIC"] = "1"
    try:
        return make()
    finally:
        os.environ.pop("DOP_FORCE_GENERIC", None)


def field(i, dtype):
    return torch.from_numpy(np.random.default_rng(i).uniform(-1, 1, CASES[i][0])).to(dtype)


def dt(case):
    return 0.02 / float(max(case[0])) ** case[1]


def scale(case):
    return 1.0 if case[1] == 2 else -1.0


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_mixed_batch_equals_generic(dtype):
    def make(us):
        return D.RK4([operator(c) for c in CASES], us, [scale(c) for c in CASES], [dt(c) for c in CASES])
    a = [field(i, dtype).to("cuda") for i in range(len(CASES))]
    b = [x.clone() for x in a]
    ra, rb = make(a), generic(lambda: make(b))
    for n in (1, 2, 3, 1):
        ra.step(n)
        rb.step(n)
        torch.cuda.synchronize()
        for c, x, y in zip(CASES, a, b):
            assert torch.isfinite(y).all()
            assert torch.equal(x, y), (c, n, (x - y).abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_mixed_classes_equal_generic(dtype):
    steps = [1 + i % 5 for i in range(len(CASES))]
    fields = [field(i, dtype).pin_memory() for i in range(len(CASES))]

    def serve():
        srv = D.Server(256 << 20)
        ids = [srv.submit(D.plan_for_shape(operator(c), c[0], dtype), f, scale(c), dt(c), n, 0.0)
               for c, f, n in zip(CASES, fields, steps)]
        srv.run()
        return [srv.results[i].clone() for i in ids]

    for c, x, y in zip(CASES, serve(), generic(serve)):
        assert torch.isfinite(y).all()
        assert torch.equal(x, y), c
