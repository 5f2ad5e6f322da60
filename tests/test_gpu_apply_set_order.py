"""GPU: terms of an apply set whose outputs others read or write in part (views of one buffer): in order,
as the same applies one by one."""
import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
from diffeqoperators_amd.apply import _padded_plan, apply_set

pytestmark = pytest.mark.gpu


class Owner:
    pass


def plan(L, out, padded):
    return _padded_plan(Owner(), [L], out, padded)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [64, 4099, 300001])
def test_a_term_that_reads_the_one_before(dtype, n):
    # the second derivative of the second derivative, in the interior of one padded buffer
    L = D.CenteredDifference(2, 4, 1.0 / (n + 1), n)
    x = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, n + 2)).to("cuda").to(dtype)
    out, ref = torch.empty(n, dtype=dtype, device="cuda"), torch.empty(n, dtype=dtype, device="cuda")
    w = torch.zeros(n + 2, dtype=dtype, device="cuda")
    p = plan(L, out, x)
    p.apply(w[1:-1], x)
    p.apply(ref, w)
    w.zero_()
    apply_set([(p, w[1:-1], x, False), (p, out, w, False)])
    assert torch.equal(out, ref)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shift", [1, 5, 2000])
def test_outputs_that_overlap(dtype, shift):
    n = 4099
    L = D.CenteredDifference(1, 4, 1.0 / (n + 1), n)
    x = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, (3, n + 2))).to("cuda").to(dtype)
    a, b = (torch.zeros(n + shift, dtype=dtype, device="cuda") for _ in range(2))
    p = plan(L, a[:n], x[0])
    terms = [(0, 0, False), (shift, 1, False), (0, 2, True)]
    for off, k, acc in terms:
        p.apply(a[off:off + n], x[k], acc)
    apply_set([(p, b[off:off + n], x[k], acc) for off, k, acc in terms])
    assert torch.equal(a, b)
