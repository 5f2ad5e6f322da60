"""The latency form of the per-point evaluation (dop_eval.hpp: shell_point, the shell of 2-D applies
and batches), compiled for the CPU, must equal the generic evaluator bit for bit at every point
of every plan it takes, and must refuse the plans outside its limits (more than two ghost taps,
periodic or per-line BCs, axes too short to keep the two ends apart)."""
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
STORAGE = {"f64": (_abi.F64, np.float64, np.uint64), "f32": (_abi.F32, np.float32, np.uint32),
           "bf16": (_abi.BF16, np.uint16, np.uint16)}


@pytest.fixture(scope="module")
def hc():
    if not os.path.exists(HC_PATH):
        pytest.skip("tests/hostcheck not built")
    L = C.CDLL(HC_PATH)
    for f in (L.hc_apply, L.hc_shell_point):
        f.argtypes = [C.POINTER(_abi.DopDesc), C.c_void_p, C.c_void_p, C.c_int]
    return L


def desc(shape, ops, Q, storage):
    js = tuple(reversed(shape))
    bcs, sem = _bcs_of(Q, len(js), js)
    return make_desc(ops, js, STORAGE[storage][0], input_kind=_abi.INPUT_GHOST, semantics=sem, bcs=bcs)


def values(shape, storage, seed):
    u = np.random.default_rng(seed).uniform(-1, 1, shape)
    if storage == "bf16":
        return (u.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return u.astype(STORAGE[storage][1])


def compare(hc, d, shape, storage):
    bits = STORAGE[storage][2]
    u = values(shape, storage, 3)
    for acc in (0, 1):
        a, b = values(shape, storage, 4), values(shape, storage, 4)
        rc = hc.hc_shell_point(C.byref(d), a.ctypes.data, u.ctypes.data, acc)
        if rc != 1:
            return rc
        assert hc.hc_apply(C.byref(d), b.ctypes.data, u.ctypes.data, acc) == 0
        np.testing.assert_array_equal(a.view(bits), b.view(bits))
    return 1


def ops_of(shape, d, a, rng, uniform, upwind):
    js = tuple(reversed(shape))
    ops = []
    for N, n in enumerate(js, 1):
        h = 1.0 / (n + 1)
        dx = h if uniform else h * (1 + 0.5 * rng.random(n + 1))
        ops.append(D.CenteredDifference[N](d, a, dx, n))
        if upwind:
            ops.append(D.UpwindDifference[N](1, 3, dx, n, rng.standard_normal(n)))
    return ops


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("bc", ["dirichlet", "neumann", "robin"])
@pytest.mark.parametrize("shape,d,a,uniform,upwind",
                         [((64, 65), 2, 4, True, False), ((61, 64), 2, 4, True, True),
                          ((64, 80), 2, 6, False, True), ((70, 64), 4, 2, True, False),
                          ((64, 64), 1, 2, True, False), ((90, 77), 3, 6, True, False),
                          ((101,), 2, 2, True, False), ((130,), 4, 8, True, False)])
def test_equal_to_generic(hc, shape, d, a, uniform, upwind, bc, storage):
    rng = np.random.default_rng(7)
    js = tuple(reversed(shape))
    atom = {"dirichlet": D.DirichletBC(0.3, -0.7), "neumann": D.NeumannBC((0.4, -0.2), 0.01, 1),
            "robin": D.RobinBC((1.0, 0.5, 0.2), (0.8, -0.4, 0.1), 0.01, 1)}[bc]
    Q = atom if len(shape) == 1 else D.compose(*D.MultiDimBC(atom, js))
    de, keep = desc(shape, ops_of(shape, d, a, rng, uniform, upwind), Q, storage)
    assert compare(hc, de, shape, storage) == 1


def test_refuses_what_it_cannot_take(hc):
    rng = np.random.default_rng(8)
    shape = (64, 64)
    ops = ops_of(shape, 2, 4, rng, True, False)
    dir0 = D.MultiDimBC[2](D.Dirichlet0BC(float), (64, 64))
    # three ghost taps; a periodic line among the x lines; a short axis
    for x in (D.MultiDimBC[1](D.RobinBC((1.0, 0.5, 0.2), (1.0, 0.5, 0.2), 0.01, 3), (64, 64)),
              D.MultiDimBC[1](D.PeriodicBC(float), (64, 64)),
              D.MultiDimBC[1](np.array([D.DirichletBC(0.0, 1.0)] * 64, dtype=object))):
        de, keep = desc(shape, ops, D.compose(x, dir0), "f64")
        assert compare(hc, de, shape, "f64") == 0
    de, keep = desc((64, 14), ops_of((64, 14), 2, 4, rng, True, False),
                    D.compose(*D.Dirichlet0BC(float, (14, 64))), "f64")
    assert compare(hc, de, (64, 14), "f64") == 0
