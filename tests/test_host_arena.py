"""The server's arena (dop_arena.hpp) over a host stand-in for the device's memory: blocks lie in what
is held and never overlap, no more than the budget is held, whatever fits the empty arena is given
(also after live requests have left it in pieces, or memory has run short), and a burst holds what it
needs, not the budget."""
import ctypes as C
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HC_PATH = os.environ.get("DOP_HOSTCHECK_LIBRARY") or os.path.join(ROOT, "tests", "hostcheck", "_build",
                                                                "libdop_hostcheck.so")
BUDGET = 1 << 22


@pytest.fixture(scope="module")
def hc():
    if not os.path.exists(HC_PATH):
        pytest.skip("tests/hostcheck not built")
    L = C.CDLL(HC_PATH)
    L.hc_arena.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int, C.POINTER(C.c_int64)]
    return L


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("limit", [1 << 40, BUDGET, BUDGET * 3 // 5])
@pytest.mark.parametrize("ahead", [0, BUDGET // 7, 4 * BUDGET, -BUDGET // 3, -4 * BUDGET])
def test_random_requests(hc, seed, limit, ahead):
    most = C.c_int64()
    assert hc.hc_arena(BUDGET, limit, ahead, 4000, seed, C.byref(most)) == 0
    assert most.value <= min(BUDGET, limit)


def test_holds_what_is_asked(hc):
    most = C.c_int64()
    assert hc.hc_arena(1 << 44, 1 << 45, 1 << 20, 0, 0, C.byref(most)) == 0
    assert most.value == 0          # nothing before the first request
