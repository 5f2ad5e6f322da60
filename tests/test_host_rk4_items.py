"""The work list of one-pass RK4 steps (dop_batch_host.cpp, dop_rk4_impl.hpp), checked on the CPU
over the sizes, orders and boundary conditions of the batch: every point belongs to exactly one patch
or marching segment, every value a patch's points read through the four stages lies in what the
patch holds, every patch fits its LDS, and every segment's cone stays on regular rows."""
import ctypes as C
import os

import numpy as np
import pytest

import diffeqoperators_amd as D
from diffeqoperators_amd import _abi
from diffeqoperators_amd.apply import _bcs_of, make_desc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HC_PATH = os.environ.get("DOP_HOSTCHECK_LIBRARY") or os.path.join(ROOT, "tests", "hostcheck", "_build",
                                                                "libdop_hostcheck.so")


@pytest.fixture(scope="module")
def hc():
    if not os.path.exists(HC_PATH):
        pytest.skip("tests/hostcheck not built")
    L = C.CDLL(HC_PATH)
    L.hc_rk4_items.argtypes = [C.POINTER(_abi.DopDesc), C.POINTER(C.c_int), C.c_void_p]
    return L


def check(hc, ops, Q, js, storage):
    bcs, sem = _bcs_of(Q, len(js), js)
    d, keep = make_desc(ops, js, storage, input_kind=_abi.INPUT_GHOST, semantics=sem, bcs=bcs)
    bad, info = C.c_int(), np.zeros(4, dtype=np.int64)
    fused = hc.hc_rk4_items(C.byref(d), C.byref(bad), info.ctypes.data)
    assert fused >= 0
    assert bad.value == 0, (bad.value, info.tolist(), js)
    return fused


@pytest.mark.parametrize("storage", [_abi.F32, _abi.F64])
@pytest.mark.parametrize("d,a", [(1, 2), (2, 2), (2, 4), (3, 4), (2, 6), (4, 4), (1, 8), (2, 8), (3, 8),
                                 (4, 8)])
def test_centered_batch(hc, d, a, storage):
    for i, n in enumerate((64, 65, 90, 128, 131, 137, 200, 257, 515, 1023, 2048)):
        for bc in (D.DirichletBC(0.1, -0.1), D.NeumannBC((0.1, 0.2), 0.01, 1),
                   D.RobinBC((1.0, 0.5, 0.1), (1.0, 0.5, -0.1), 0.01, 1)):
            h = 1.0 / (n + 1)
            check(hc, [D.CenteredDifference(d, a, h, n)], bc, (n,), storage)
            if n > 515 and bc.a_l.size != 1:
                continue
            m = n if i % 2 else n + 3 * i
            ops = [D.CenteredDifference[1](d, a, h, n), D.CenteredDifference[2](d, a, h, m)]
            fused = check(hc, ops, D.compose(*D.MultiDimBC(bc, (n, m))), (n, m), storage)
            if min(n, m) >= 200 and not (storage == _abi.F64 and a == 8):
                assert fused == 2


@pytest.mark.parametrize("storage", [_abi.F32, _abi.F64])
def test_long_lines_and_other_windows(hc, storage):
    rng = np.random.default_rng(3)
    for n in (65536, 40001):
        for d, a in ((4, 8), (2, 4), (3, 2)):
            assert check(hc, [D.CenteredDifference(d, a, 1.0 / (n + 1), n)], D.DirichletBC(0.0, 1.0), (n,),
                         storage) == 1
    for js in ((150, 400), (70, 300), (301, 140)):
        ops = []
        for N, n in enumerate(js, 1):
            dx = (1 + 0.5 * rng.random(n + 1)) / n
            ops += [D.CenteredDifference[N](2, 2 if N == 1 else 6, dx, n),
                    D.UpwindDifference[N](1, 3, dx, n, rng.standard_normal(n))]
        check(hc, ops, D.compose(*D.Dirichlet0BC(float, js)), js, storage)
        # one axis's window one-sided, the other's wider
        ops = [D.UpwindDifference[1](1, 3, 1.0 / js[0], js[0], 1.0), D.CenteredDifference[2](2, 6, 1.0 / js[1], js[1])]
        check(hc, ops, D.compose(*D.Dirichlet0BC(float, js)), js, storage)
