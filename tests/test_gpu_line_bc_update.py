"""GPU: dop_plan_update of a 3-D plan with one BC per line.  The shell of a plan whose lines are all
affine reads each x line's ends only; lines that the update would make periodic read their far end, so
it is refused, as for any other change of the BCs' kinds, and the plan keeps its values.  Lines made
affine, and other values, are taken."""
import numpy as np
import pytest
import torch

import diffeqoperators_amd as D
from diffeqoperators_amd import _abi
from diffeqoperators_amd.apply import Plan, _ghost_descs, _ghost_terms
from test_host_line_bcs import bc_array

pytestmark = pytest.mark.gpu

SHAPE = (24, 20, 70)


def operator(seed, periodic):
    rng = np.random.default_rng(11)
    js = tuple(reversed(SHAPE))
    ops = [D.CenteredDifference[N](2, 4, 0.05 * (1 + 0.5 * rng.random(n + 1)), n) for N, n in enumerate(js, 1)]
    rng = np.random.default_rng(seed)
    Qs = [D.MultiDimBC[N](bc_array(rng, tuple(js[k] for k in range(3) if k != N - 1), 0.05,
                                   periodic if N == 1 else 0.0)) for N in (1, 2, 3)]
    return sum(ops[1:], ops[0]) * D.compose(*Qs)


def desc(A, u):
    (d, keep, _), = _ghost_descs(_ghost_terms(A), u, _abi.ACC_AUTO)
    return d, keep


def test_lines_made_periodic_are_refused():
    u = torch.from_numpy(np.random.default_rng(3).uniform(-1, 1, SHAPE)).to("cuda")
    out, ref = torch.empty_like(u), torch.empty_like(u)

    def fresh(A):
        D.plans_for(A, u)[0].apply(ref, u)
        return ref
    a, b, mixed = operator(1, 0.0), operator(2, 0.0), operator(3, 0.5)
    p = Plan(*desc(a, u))
    p.update(*desc(b, u))
    p.apply(out, u)
    assert torch.equal(out, fresh(b))
    with pytest.raises(_abi.DopError) as e:
        p.update(*desc(mixed, u))
    assert e.value.code == _abi.EINVAL
    p.apply(out, u)
    assert torch.equal(out, fresh(b))
    q = Plan(*desc(mixed, u))
    q.update(*desc(a, u))
    q.apply(out, u)
    assert torch.equal(out, fresh(a))
