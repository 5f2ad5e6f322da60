"""GPU: RK4 steps in one pass over the grid (dop_rk4_impl.hpp) against the same steps taken stage by
stage.  A plan created for the generic kernel has no tiles, so its steps run every stage over the
whole grid; the one-pass steps, their rims and the copy back must give the same state bit for
bit, after odd and even numbers of steps, at grids around the edges of segments and chunks, for
every window width, accumulator and grid kind; a grid too small for a box is stage-wise in both."""
import os

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu


def operator(shape, d, a, rng_seed, uniform, upwind):
    rng = np.random.default_rng(rng_seed)
    js = tuple(reversed(shape))
    ops = []
    for N, n in enumerate(js, 1):
        h = 1.0 / (n + 1)
        dx = h if uniform else h * (1 + 0.3 * rng.random(n + 1))
        ops.append(D.CenteredDifference[N](d, a, dx, n))
        if upwind:
            ops.append(D.UpwindDifference[N](1, 3, dx, n, rng.standard_normal(n)))
    A = ops[0]
    for L in ops[1:]:
        A = A + L
    return A * D.compose(*D.RobinBC((1.0, 0.5, 0.1), (1.0, 0.5, -0.2),
                                    tuple(1.0 / (n + 1) for n in js), 1, js))


def stagewise(make):
    os.environ["DOP_FORCE_GENERIC"] = "1"
    try:
        return make()
    finally:
        os.environ.pop("DOP_FORCE_GENERIC", None)


CASES = [((140, 140), 2, 2, True, False), ((150, 257), 2, 4, True, False),
         ((131, 470), 2, 4, False, True), ((300, 161), 2, 6, True, False),
         ((160, 520), 4, 2, True, False), ((170, 180), 2, 8, True, False),
         ((175, 290), 4, 8, True, False), ((200, 333), 3, 4, False, False),
         ((96, 300), 2, 4, True, False), ((1030, 1026), 2, 4, True, True)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_one_pass_equals_stagewise(dtype):
    fields = [torch.from_numpy(np.random.default_rng(i).uniform(-1, 1, c[0])).to("cuda").to(dtype)
              for i, c in enumerate(CASES)]
    scale = [-1.0 if c[1] % 2 else (1.0 if c[1] == 2 else -1.0) for c in CASES]
    dts = [0.02 / float(max(c[0])) ** c[1] for c in CASES]

    def integrator(us):
        return D.RK4([operator(c[0], c[1], c[2], i, c[3], c[4]) for i, c in enumerate(CASES)], us,
                     scale, dts)

    a, b = [f.clone() for f in fields], [f.clone() for f in fields]
    ra, rb = integrator(a), stagewise(lambda: integrator(b))
    for n in (1, 2, 3, 1):
        ra.step(n)
        rb.step(n)
        torch.cuda.synchronize()
        for c, x, y in zip(CASES, a, b):
            assert torch.isfinite(y).all()
            assert torch.equal(x, y), (c, n, (x - y).abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_served_odd_and_even_steps_equal_stagewise(dtype):
    cases = [CASES[1], CASES[2], CASES[5], CASES[8], CASES[9]]
    steps = [3, 4, 1, 2, 5]
    fields = [torch.from_numpy(np.random.default_rng(i).uniform(-1, 1, c[0])).to(dtype).pin_memory()
              for i, c in enumerate(cases)]

    def serve():
        srv = D.Server(256 << 20)
        plans = [D.plan_for_shape(operator(c[0], c[1], c[2], i, c[3], c[4]), c[0], dtype)
                 for i, c in enumerate(cases)]
        for i, (c, p, f, n) in enumerate(zip(cases, plans, fields, steps)):
            srv.submit(p, f, 1.0, 0.02 / float(max(c[0])) ** 2, n, 0.0)
        srv.run()
        return [srv.results[i].clone() for i in range(len(cases))]

    for x, y in zip(serve(), stagewise(serve)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_patches_of_mixed_windows_equal_stagewise(dtype):
    # windows of different widths per axis (regular rows outside the tiles' box, taps the wider
    # window adds with weight 0), 1-D grids of one and several patches, far patch origins
    shapes = [((140, 151), (2, 6)), ((180, 97), (6, 2)), ((230, 333), (4, 2)), ((64, 70), (2, 4)),
              ((66,), (2,)), ((1025,), (6,)), ((65536,), (4,)), ((40000,), (8,))]

    def make(us):
        ops = []
        for shape, orders in shapes:
            js = tuple(reversed(shape))
            A = None
            for N, (n, a) in enumerate(zip(js, orders), 1):
                L = D.CenteredDifference[N](2, a, 1.0 / (n + 1), n)
                A = L if A is None else A + L
            dx = tuple(1.0 / (n + 1) for n in js)
            robin = ((1.0, 0.5, 0.1), (1.0, 0.5, -0.2))
            if len(js) == 1:
                ops.append(A * D.RobinBC(*robin, dx[0], 1))
            else:
                ops.append(A * D.compose(*D.RobinBC(*robin, dx, 1, js)))
        return D.RK4(ops, us, [1.0] * len(us), [0.02 / max(s) ** 2 for s, _ in shapes])

    fields = [torch.from_numpy(np.random.default_rng(i).uniform(-1, 1, s)).to("cuda").to(dtype)
              for i, (s, _) in enumerate(shapes)]
    a, b = [f.clone() for f in fields], [f.clone() for f in fields]
    ra, rb = make(a), stagewise(lambda: make(b))
    for n in (1, 2):
        ra.step(n)
        rb.step(n)
        torch.cuda.synchronize()
        for c, x, y in zip(shapes, a, b):
            assert torch.isfinite(y).all()
            assert torch.equal(x, y), (c, n, (x - y).abs().max().item())
