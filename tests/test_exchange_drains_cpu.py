"""The solves on the chip reuse an exchange's words three rounds after the round
that filled them: a workgroup empties its words of round r - 1 in round r, and a
peer that has passed round r + 2 looks at them again.  What makes the empty words
visible by then is a drain of the stores (peer_drain) between a workgroup's
round r and its publication in round r + 2.  That cannot be shown on the device
(the words almost always arrive in time), so the order of drains and exchanges is
read from the sources, over every path through the loops."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "elastic_amd", "csrc")


def _block(text, start):
    """The text between the braces that open at or after `start`."""
    i = text.index("{", start)
    depth = 0
    for j in range(i, len(text)):
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        if depth == 0:
            return text[i + 1:j], j + 1
    raise AssertionError("unbalanced braces")


def _paths(body):
    """Every order of 'D' (drain) and 'X' (exchange) in a loop body: a block with
    exchanges after an `if` is taken or not, a loop of two passes runs twice."""
    head = re.compile(r"peer_drain\(\)|(?:res|gm)_exchange<|for \(int pass = 0; pass < 2[^{]*|"
                      r"\bif \(!\(n2 > [^{;]*")
    paths, at = [""], 0
    while True:
        m = head.search(body, at)
        if not m:
            return paths
        t = m.group(0)
        if t.startswith("for") or t.startswith("if"):
            inner, at = _block(body, m.end())
            sub = _paths(inner)
            tails = [a + b for a in sub for b in sub] if t.startswith("for") else [""] + sub
            paths = [p + q for p in paths for q in tails]
        else:
            paths = [p + ("D" if t.startswith("peer") else "X") for p in paths]
            at = m.end()


def _undrained(steps):
    """First round r of the sequence without a drain before round r + 2 publishes."""
    at = [k for k, c in enumerate(steps) if c == "X"]
    for r in range(len(at) - 2):
        if "D" not in steps[at[r]:at[r + 2]]:
            return r
    return None


@pytest.mark.parametrize("name,rounds", [("pcg_resident.h", {2}), ("bicgstab_resident.hip", {4}),
                                         ("gmres_resident.hip", {2, 3})])
def test_every_word_is_visibly_empty_before_its_next_round(name, rounds):
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())
    body, _ = _block(text, text.index("while (true)"))
    paths = _paths(body)
    assert {p.count("X") for p in paths} == rounds, paths
    for a in paths:
        for b in paths:
            for c in paths:
                assert _undrained(a + b + c) is None, (a, b, c)


def test_the_check_finds_a_missing_drain():
    assert _undrained("DXXDXX") is None
    assert _undrained("DXXX") == 0 and _undrained("XXDXXX") == 2


def test_a_lost_word_is_told_behind_a_barrier():
    """In a batch's step, whose workgroups go on to the next instance, the
    flag that a wait ran out changes only where every wavefront reads the same: in
    an exchange before its last barrier, or behind a barrier that follows it.  (Set
    earlier, a slow wavefront would see it as the exchange's and leave the loop alone,
    one barrier off from the others.)"""
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "pcg_resident.h")).read())
    # the form of a batch's step
    text, n = re.subn(r"if constexpr \(STEP\) (sh\.late = 1;)\s*else sh\.bad = 1;", r"\1", text)
    assert n == 1
    body, _ = _block(text, text.index("while (true)"))
    marks = re.findall(r"res_exchange<|__syncthreads\(\)|sh\.bad = 1", body)
    assert marks.count("sh.bad = 1") == 1
    for k, m in enumerate(marks):
        if m == "sh.bad = 1":
            assert marks[k - 1] == "__syncthreads()", marks
