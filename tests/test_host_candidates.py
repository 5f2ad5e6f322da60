"""Which tile shapes the tuner tries (dop_fast.cpp: fast_candidate): 3-D chunks of 16 planes only where
chunks of 32 leave fewer than four blocks per CU; every other shape always."""
import ctypes as C
import os

import pytest

import diffeqoperators_amd as D
from diffeqoperators_amd import _abi
from diffeqoperators_amd.apply import _bcs_of, make_desc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HC_PATH = os.environ.get("DOP_HOSTCHECK_LIBRARY") or os.path.join(ROOT, "tests", "hostcheck", "_build",
                                                                "libdop_hostcheck.so")


@pytest.mark.parametrize("storage", [_abi.F32, _abi.F64, _abi.BF16])
@pytest.mark.parametrize("n", [64, 200, 512])
def test_short_chunks(n, storage):
    if not os.path.exists(HC_PATH):
        pytest.skip("tests/hostcheck not built")
    L = C.CDLL(HC_PATH)
    ip = C.POINTER(C.c_int)
    L.hc_candidate.argtypes = [C.POINTER(_abi.DopDesc), C.c_int, ip, ip, ip]
    ops = [D.CenteredDifference[N](2, 6, 1.0 / (n + 1), n) for N in (1, 2, 3)]
    bcs, sem = _bcs_of(D.compose(*D.Dirichlet0BC(float, (n, n, n))), 3, (n, n, n))
    d, keep = make_desc(ops, (n, n, n), storage, input_kind=_abi.INPUT_GHOST, semantics=sem, bcs=bcs)
    chunk, rows, vx = C.c_int(), C.c_int(), C.c_int()
    count = skipped = 0
    while True:
        tried = L.hc_candidate(C.byref(d), count, C.byref(chunk), C.byref(rows), C.byref(vx))
        if tried < 0:
            break
        box = n - 4     # (rows with windows of 7 points; along x less)
        blocks = -(-box // (64 * vx.value)) * -(-box // rows.value) * -(-box // 32)
        assert tried == (chunk.value != 16 or blocks < 1024), (count, chunk.value, rows.value, vx.value)
        skipped += not tried
        count += 1
    assert count == 36 and (skipped > 0) == (n == 512)
