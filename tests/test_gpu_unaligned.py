"""GPU: u and du at any element offset go through the tiles (element-aligned vector loads and stores)
and give the generic kernel's values bit for bit, touching nothing beside du."""
import os

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(130, 259), (41, 47, 301)])
@pytest.mark.parametrize("offs", [(1, 0), (0, 1), (3, 5)])
def test_any_element_offset(dtype, shape, offs):
    js = tuple(reversed(shape))
    A = None
    for N, n in enumerate(js, 1):
        L = D.CenteredDifference[N](2, 4, 1.0 / (n + 1), n)
        A = L if A is None else A + L
    A = A * D.compose(*D.RobinBC((1.0, 0.5, 0.1), (1.0, 0.5, -0.2), tuple(1.0 / (n + 1) for n in js), 1, js))
    total = int(np.prod(shape))
    x = torch.from_numpy(np.random.default_rng(7).uniform(-1, 1, total)).to("cuda").to(dtype)
    bu = torch.zeros(total + 8, dtype=dtype, device="cuda")
    bd = torch.zeros(total + 8, dtype=dtype, device="cuda")
    u, du = bu[offs[0]:offs[0] + total], bd[offs[1]:offs[1] + total]
    u.copy_(x)
    D.plan_for_shape(A, shape, dtype).apply(du, u)
    os.environ["DOP_FORCE_GENERIC"] = "1"
    try:
        ref = torch.empty_like(x)
        D.plan_for_shape(A, shape, dtype).apply(ref, x)
    finally:
        os.environ.pop("DOP_FORCE_GENERIC", None)
    assert torch.equal(du, ref)
    assert (bd[:offs[1]] == 0).all() and (bd[offs[1] + total:] == 0).all()
