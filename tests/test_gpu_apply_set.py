"""GPU: gradient, divergence and curl through one launch for all terms (dop_apply_set) against the
same terms applied one by one: the same sums in the same order, so the same values bit for bit, at
extents around whole groups of four points, with one-sided rows at the edges of every axis."""
import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
from diffeqoperators_amd import vector_calculus as vc

pytestmark = pytest.mark.gpu


def one_by_one(monkeypatch, f):
    with monkeypatch.context() as m:
        m.setattr(vc, "apply_set", lambda terms: [p.apply(du, u, a) for p, du, u, a in terms])
        return f()


SHAPES = [(9,), (10,), (4099,), (9, 10), (33, 12), (70, 263), (9, 9, 9), (10, 11, 13), (16, 12, 20),
          (21, 34, 67), (47, 38, 125), (260, 66, 131),
          (90, 98, 250), (48, 470, 101)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("a", [2, 4, 6])
@pytest.mark.parametrize("uniform", [True, False])
def test_one_launch_equals_launches_in_order(monkeypatch, dtype, a, uniform):
    rng = np.random.default_rng(a)
    for shape in SHAPES:
        js = tuple(reversed(shape))
        dx = tuple(0.1 if uniform else 0.05 * (1 + 0.5 * rng.random(n + 1)) for n in js)
        f = torch.from_numpy(rng.uniform(-1, 1, (len(js),) + tuple(s + 2 for s in shape)))
        f = f.to("cuda").to(dtype)
        ops = [(D.Gradient(a, dx, js), f[0]), (D.Divergence(a, dx, js), f)]
        if len(js) == 3 and js[0] == js[1] == js[2]:
            ops.append((D.Curl(a, dx, js), f))
        for A, u in ops:
            got, ref = A * u, one_by_one(monkeypatch, lambda: A * u)
            assert torch.isfinite(ref).all()
            assert torch.equal(got, ref), (shape, type(A).__name__)


@pytest.mark.parametrize("n", [24, 31, 97, 140, 157])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("a", [2, 4, 6])
def test_curl_equals_launches_in_order(monkeypatch, n, dtype, a):
    u = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, (3, n + 2, n + 2, n + 2)))
    u = u.to("cuda").to(dtype)
    A = D.Curl(a, (0.1, 0.2, 0.3), (n, n, n))
    assert torch.equal(A * u, one_by_one(monkeypatch, lambda: A * u))
