"""GPU: every tile-shape candidate of the tiled path, bit for bit against the generic kernel, with
the candidate that was asked for shown to be the one that ran: an index beyond the candidates is
ignored when a plan is made, so a sweep that only counts too far passes on the default one."""
import pytest
import torch

from test_gpu_tiled import build, generic_of, plan_with_variant

pytestmark = pytest.mark.gpu


def candidates(shape, dtype):
    """dop_fast.cpp, fast_variant_count: rows of at least 32 points take 16-byte loads (VX points), 2-D
    rows of at least 256 VX points also twice that."""
    vx = 2 if dtype == torch.float64 else 4
    if len(shape) == 2:
        return 64 if shape[-1] >= 256 * vx else 32
    return 36 if shape[-1] >= 32 else 18


# window half-widths below and above the points per lane (edge-loaded and overlapping segments),
# rows that are whole groups and rows that are not, twice the points per lane among both
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape,kh", [((40, 1407), 2), ((36, 1001), 1), ((33, 611), 3), ((45, 1101), 5),
                                      ((38, 1038), 4), ((300, 263), 2), ((50, 24), 1), ((41, 1040), 3),
                                      ((21, 45, 267), 4), ((40, 72, 101), 3), ((23, 38, 134), 2),
                                      ((19, 33, 28), 1), ((21, 45, 532), 3)])
def test_every_candidate_bitwise(shape, kh, dtype):
    A, u = build(shape, kh, dtype, seed=5, uniform=False, upwind=(kh == 3))
    ref = torch.empty_like(u)
    generic_of(A, u).apply(ref, u)
    n = candidates(shape, dtype)
    for v in range(n):
        print(f"case: variant {v} {shape} {dtype}", flush=True)
        plan = plan_with_variant(A, u, v)
        assert plan.variant[0] == v
        out = torch.empty_like(u)
        plan.apply(out, u)
        assert torch.equal(out, ref), v
    assert plan_with_variant(A, u, n).variant[0] < n     # there is no further one
