"""The pool of plans that owners have left (apply.py), with stand-ins for the plans: which set a search
takes, what the pool holds in number and in bytes, and owners that go in the middle of a search."""
import pytest

import diffeqoperators_amd.apply as ap


class Plan:
    def __init__(self, name, device_bytes=1):
        self.name, self.device_bytes = name, device_bytes


@pytest.fixture(autouse=True)
def pool():
    kept = list(ap._POOL)
    ap._POOL.clear()
    ap._pool_held = 0
    yield ap._POOL
    ap._POOL.clear()
    ap._pool_held = 0
    for e in kept:
        ap._pool_put(e[0], e[1], e[2])


def names():
    return [e[1][0].name for e in ap._POOL]


def test_newest_of_structure_and_stream():
    for name, skey, stream in (("a", 1, 7), ("b", 1, 8), ("c", 2, 7), ("d", 1, 7), ("e", 2, 8)):
        ap._pool_put(skey, [Plan(name)], stream)
    assert ap._pool_take(3, 7) is None and names() == ["a", "b", "c", "d", "e"]
    assert ap._pool_take(1, 7)[0].name == "d" and names() == ["a", "b", "c", "e"]
    assert ap._pool_take(1, 7)[0].name == "a" and names() == ["b", "c", "e"]
    assert ap._pool_take(1, 7) is None
    assert ap._pool_held == 3


def test_bounded_in_number_and_bytes():
    for k in range(100):
        ap._pool_put(1, [Plan(k)], 0)
    assert names() == list(range(36, 100))
    third = ap._POOL_BYTES // 3
    for k in range(5):
        ap._pool_put(2, [Plan(k, third)], 0)
    assert names() == [2, 3, 4] and ap._pool_held == 3 * third
    ap._pool_put(2, [Plan("long", 5 * third)], 0)      # the newest stays, whatever it holds
    assert names() == ["long"] and ap._pool_held == 5 * third
    ap._pool_put(2, [Plan("x")], 0)
    assert names() == ["x"] and ap._pool_held == 1
    assert ap._pool_take(2, 0)[0].name == "x" and ap._pool_held == 0 and not ap._POOL


@pytest.mark.parametrize("big", [0, 1 << 40])
def test_an_owner_that_goes_during_a_search(big):
    class Key:
        def __eq__(self, other):        # as a collection in the middle of the search would
            ap._pool_put("left", [Plan("left", 1 + big)], 0)
            return False
    for k in range(64):
        ap._pool_put(k, [Plan(k)], 0)
    assert ap._pool_take(Key(), 0) is None
    assert 1 <= len(ap._POOL) <= 64
    assert ap._pool_held == sum(e[3] for e in ap._POOL)
