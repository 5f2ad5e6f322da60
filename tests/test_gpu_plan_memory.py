"""GPU: what the plans that owners have left hold of the device's memory: long non-uniform lines have
tables of tens of megabytes a plan."""
import gc

import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
import diffeqoperators_amd.apply as ap

pytestmark = pytest.mark.gpu


def test_pool_is_bounded_in_bytes():
    n, count = 1 << 20, 24
    dx = (1.0 + 0.1 * np.random.default_rng(5).random(n + 1)) / n
    L = D.CenteredDifference(2, 2, dx, n)
    u = torch.from_numpy(np.random.default_rng(6).uniform(-1, 1, n)).to("cuda")
    one = D.plans_for(L * D.DirichletBC(0.0, 1.0), u)[0].device_bytes
    assert count * one > 2 * ap._POOL_BYTES              # or the test says nothing
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    out = torch.empty_like(u)
    owners = [L * D.DirichletBC(0.1 * k, 1.0) for k in range(count)]
    for A in owners:
        D.mul_(out, A, u)
    del owners, A
    gc.collect()
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < ap._POOL_BYTES + one + (64 << 20)
    want = torch.empty_like(u)
    for g in (5.0, 6.0):                                 # what is left is still good for the next
        D.plans_for(L * D.DirichletBC(g, 1.0), u)[0].apply(want, u)
        assert torch.equal(D.mul_(out, L * D.DirichletBC(g, 1.0), u), want)
