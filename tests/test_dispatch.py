"""The rules that pick a kernel's form (csrc/bssn_dispatch.h), compiled by the host compiler:
wave-private bricks wherever the shared ones were measured slower, and the other way round."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "integer-schemes_amd" / "csrc"

CHECK = r"""
#include <cstdio>
#include "bssn_dispatch.h"
int main() {
  char what[16];
  int ord;
  long waves, groups;
  while (std::scanf("%15s %d %ld %ld", what, &ord, &waves, &groups) == 4)
    std::printf("%d\n", (int)bssn::RULE);
}
"""


def ask(tmp_path, rule, rows):
    """The rule's answers for rows of (what, order, wave-private bricks, shared bricks)."""
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(CHECK.replace("RULE", rule))
    subprocess.run([cxx, "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    text = "".join(" ".join(map(str, r)) + "\n" for r in rows)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
    return [bool(int(v)) for v in out.stdout.split()]


def bricks(n, e):
    return -(-n[0] // e[0]) * -(-n[1] // e[1]) * -(-n[2] // e[2])


def row(what, order, n, copies=1):
    return what + "+" * (copies > 1), order, copies * bricks(n, (4, 4, 4)), copies * bricks(n, (4, 4, 16))


# points of one launch, copies of them in a batch, and whether shared bricks were the faster form
# there: (FD4 RHS, FD4 step, FD6 RHS, FD6 step, FD8 RHS, FD8 step), the RHS bare, the step with
# Kreiss-Oliger terms; None: within 2 %, or the two
# forms not timed there
FUSED = [
    ((256, 256, 4), 1, (0, 0, 0, 0, 0, 0)), ((256, 256, 8), 1, (0, 0, 0, 0, None, 1)),
    ((160, 160, 8), 1, (0, 0, 0, 0, 1, 1)), ((100, 100, 8), 1, (0, 0, None, 0, 1, 1)),
    ((160, 160, 20), 1, (0, 1, 1, 1, 1, 1)), ((200, 200, 20), 1, (0, 1, 1, 1, 1, 1)),
    ((48, 48, 56), 1, (0, 0, 1, 0, 1, 1)), ((45, 45, 52), 1, (0, 0, 1, 0, 1, 1)),
    ((103, 66, 33), 1, (0, None, 1, 1, 1, 1)), ((39, 82, 75), 1, (1, 1, 1, 1, 1, 1)),
    ((72, 72, 8), 1, (0, 0, 0, 0, 0, 0)), ((40, 40, 40), 1, (0, 0, 0, 0, 0, 0)),
    ((48, 48, 48), 1, (1, 1, 1, 1, 1, 1)), ((64, 64, 20), 1, (1, 1, 1, 1, 1, 1)),
    ((90, 90, 49), 1, (1, 1, 1, 1, 1, 1)), ((256, 256, 256), 1, (1, 1, 1, 1, 1, 1)),
    ((15, 15, 19), 400, (0, None, None, None, None, None)),
    ((9, 9, 13), 400, (None, 1, None, 1, None, 1)), ((8, 8, 8), 500, (None, 0, None, 0, None, 0)),
    ((38, 38, 20), 60, (0, None, None, None, None, None)),
    ((22, 22, 22), 17, (1, None, None, None, None, None)),
]


def test_fused_form(tmp_path):
    rows, want = [], []
    for n, copies, faster in FUSED:
        for i, shared in enumerate(faster):
            if shared is not None:
                rows.append(row(("bare", "step")[i % 2], (4, 6, 8)[i // 2], n, copies))
                want.append(bool(shared))
    got = ask(tmp_path, "fused_shared(ord, what[0] == 'b', what[0] == 's', what[4] == '+', waves, groups)", rows)
    assert got == want, [(r, w) for r, w, g in zip(rows, want, got) if g != w]


# (FD4, FD6, FD8) of the constraints
CONSTRAINTS = [
    ((12, 12, 12), (0, 0, None)), ((24, 24, 24), (0, 0, None)), ((32, 32, 32), (0, 0, None)),
    ((40, 40, 40), (0, 0, 0)), ((64, 64, 12), (0, 1, 1)), ((64, 64, 16), (0, 1, 1)),
    ((48, 48, 48), (1, 1, 1)), ((48, 48, 56), (0, None, 1)), ((103, 66, 33), (0, 1, 1)),
    ((39, 82, 75), (1, 1, 1)), ((128, 128, 24), (1, 1, 1)), ((160, 160, 8), (0, 0, 0)),
    ((256, 256, 8), (0, 0, 0)), ((256, 256, 4), (0, 0, 0)), ((150, 150, 150), (1, 1, 1)),
]


def test_constraints_form(tmp_path):
    rows = [row("c", order, n) for n, faster in CONSTRAINTS
            for order, shared in zip((4, 6, 8), faster) if shared is not None]
    want = [bool(v) for _, faster in CONSTRAINTS for v in faster if v is not None]
    got = ask(tmp_path, "constraints_shared(ord, waves, groups)", rows)
    assert got == want, [(r, w) for r, w, g in zip(rows, want, got) if g != w]


# (FD4 fp64, FD4 BFP32, FD6 fp64, FD6 BFP32) of the derivative bundle
BUNDLE = [
    ((12, 12, 12), (1, 1, 1, 1)), ((40, 40, 40), (1, 1, 1, 1)), ((128, 128, 128), (1, 1, 1, 1)),
    ((72, 72, 8), (1, 1, 1, 1)), ((100, 100, 8), (None, 0, 1, 1)), ((160, 160, 8), (1, 0, 0, 0)),
    ((256, 256, 8), (1, 0, 0, 0)), ((256, 256, 4), (0, 0, 0, 0)), ((200, 200, 20), (1, 1, 1, 1)),
    ((96, 96, 12), (1, 1, 1, 1)),
]


def test_bundle_form(tmp_path):
    rows, want = [], []
    for n, faster in BUNDLE:
        for i, shared in enumerate(faster):
            if shared is not None:
                rows.append(row(("fp64", "bfp")[i % 2], (4, 6)[i // 2], n))
                want.append(bool(shared))
    got = ask(tmp_path, "bundle_shared(ord, what[0] == 'f', waves, groups)", rows)
    assert got == want, [(r, w) for r, w, g in zip(rows, want, got) if g != w]
