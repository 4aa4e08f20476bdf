"""solv compares the caller's pattern with the one its context holds.  A structure
that the library fails to build (out of memory) leaves the context without any, so
neither that pattern nor the one before it is the context's: the next call sets its
structure first.  The context is a stand-in that keeps the library's rules (values
need a structure; one that fails drops the one before)."""
import numpy as np
import pytest

from elastic_amd import _lib, solver


class _Held:
    def __init__(self):
        self.pattern, self.calls = None, []

    def set_structure(self, ia, ja):
        self.calls.append("structure")
        self.pattern = None
        if ja.size and ja.max() > 4:
            raise _lib.ElasticError(_lib.OOM, "device memory")
        self.pattern = (ia.copy(), ja.copy())

    def set_values(self, ad, al):
        self.calls.append("values")
        if self.pattern is None:
            raise _lib.ElasticError(_lib.NOT_READY, "structure not set")
        self.used = (self.pattern[1].copy(), np.array(al))

    def solve(self, b, **kw):
        return np.array(b), {}


PATTERNS = {"first": [1, 1, 2], "second": [1, 2, 3], "failing": [1, 2, 9], "longer": [1, 1, 2, 3]}


def _call(name):
    ja = np.array(PATTERNS[name], np.int32)
    neq = 4
    ia = np.array([1, 1, 2, 3, 1 + len(ja)], np.int32)
    x = np.zeros(neq)
    solver.solv(neq, len(ja), ia, ja, np.ones(neq), np.arange(1.0, 1 + len(ja)), np.zeros(neq),
                np.ones(neq), x)
    return ja


@pytest.mark.parametrize("before", ["first", "longer"])
@pytest.mark.parametrize("after", ["first", "second", "longer"])
def test_a_structure_that_fails_does_not_stand_in_the_way(monkeypatch, before, after):
    c = _Held()
    monkeypatch.setattr(solver, "_default_ctx", c)
    _call(before)
    with pytest.raises(_lib.ElasticError):
        _call("failing")
    ja = _call(after)
    assert np.array_equal(c.used[0], ja) and len(c.used[1]) == len(ja)


def test_patterns_of_the_same_sizes_are_told_apart(monkeypatch):
    c = _Held()
    monkeypatch.setattr(solver, "_default_ctx", c)
    for name in ("first", "second", "second", "first"):
        ja = _call(name)
        assert np.array_equal(c.used[0], ja)
    assert c.calls.count("structure") == 3
