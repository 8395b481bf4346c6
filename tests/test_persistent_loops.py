"""Loops whose waves take work from a counter: the value of an atomic that only
some lanes of a wave execute is not broadcast to the others inside a loop.

The branch around such an atomic stands beside the loop's back edge, where one
wave's lanes can be split across iterations; the lanes left without the atomic
then go on with a value that is no item's.  Every lane issues the atomic instead
(eval_device.hpp lane_slot)."""
import glob
import os
import re

from helpers import ROOT

SOURCES = sorted(glob.glob(os.path.join(ROOT, "xray_projection_render_amd", "csrc", "*.h*")))
LANE = re.compile(r"if\s*\([^;{}]*(?:lane|threadIdx)[^;{}]*\)\s*$")
LOOP = re.compile(r"\b(?:for|while)\s*\(|\bdo\s*$")


def _plain(text):
    """Without comments."""
    text = re.sub(r"/\*.*?\*/", " ", text, flags=re.S)
    return re.sub(r"//[^\n]*", "", text)


def lane_atomics_in_loops(text):
    """Statements `x = atomicAdd(...)` under a condition on the lane, inside a
    loop's braces."""
    text, heads, found, start = _plain(text), [], [], 0
    for i, c in enumerate(text):
        if c in "{};":
            head = text[start:i]
            if c == ";" and re.search(r"=\s*atomic\w+\s*\(", head):
                # the statement's own condition, or that of the block it is in
                own = LANE.search(head[:re.search(r"\w+\s*=\s*atomic", head).start()])
                block = heads and LANE.search(heads[-1])
                outer = heads[:-1] if block else heads
                if (own or block) and any(LOOP.search(h) for h in outer):
                    found.append(" ".join(head.split()))
            if c == "{":
                heads.append(head.strip())
            elif c == "}" and heads:
                heads.pop()
            # a for's own semicolons do not end a head
            if not (c == ";" and head.count("(") > head.count(")")):
                start = i + 1
    return found


def test_the_check_finds_the_form():
    bad = "void f() { for (;;) { unsigned t = 0; if (lane == 0) t = atomicAdd(p, 1u); use(t); } }"
    block = "void f() { while (go) { if ((threadIdx.x & 63) == 0) { t = atomicAdd(p, 1u); } } }"
    once = "void f() { if (lane == 0) t = atomicAdd(p, 1u); for (int i = 0; i < n; ++i) { g(i); } }"
    every = "void f() { for (;;) { t = atomicAdd(lane_slot(p, s), first_lane() ? 1u : 0u); } }"
    assert lane_atomics_in_loops(bad) and lane_atomics_in_loops(block)
    assert not lane_atomics_in_loops(once) and not lane_atomics_in_loops(every)


def test_no_loop_broadcasts_a_lane_conditional_atomic():
    assert SOURCES
    bad = {os.path.basename(p): lane_atomics_in_loops(open(p).read()) for p in SOURCES}
    assert not {p: f for p, f in bad.items() if f}
