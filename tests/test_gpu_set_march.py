"""GPU: gradient and divergence over boxes large enough for the marching form at every window that it
has (dop_set.hip: 2^21 points of the box where all terms' rows are regular), with rows of odd length,
against the terms applied one by one: bit for bit."""
import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
from test_gpu_apply_set import one_by_one

pytestmark = pytest.mark.gpu

MARCH_POINTS = 1 << 21


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("a", [2, 4, 6])
@pytest.mark.parametrize("shape", [(265, 70, 133), (75, 181, 181), (52, 300, 158)])
def test_marching_equals_launches_in_order(monkeypatch, shape, a, dtype):
    js = tuple(reversed(shape))
    box = [n - (a - 2) for n in js]      # rows whose window of a + 1 points is centered
    assert np.prod(box) >= MARCH_POINTS and min(box) >= 32
    f = torch.from_numpy(np.random.default_rng(a).uniform(-1, 1, (3,) + tuple(s + 2 for s in shape)))
    f = f.to("cuda").to(dtype)
    for A, u in ((D.Gradient(a, (0.1, 0.2, 0.3), js), f[0]), (D.Divergence(a, (0.1, 0.2, 0.3), js), f)):
        got, ref = A * u, one_by_one(monkeypatch, lambda: A * u)
        assert torch.isfinite(ref).all()
        assert torch.equal(got, ref), type(A).__name__
