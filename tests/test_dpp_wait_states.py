"""Cross-lane (DPP) operands of inline assembly: the wait states stand in the statement that reads the operand.

A DPP instruction must not read a register that a vector instruction wrote in the two wait states before it.  The
compiler keeps that distance for its own instructions, not into inline assembly, and it may put a copy or a reload of
an operand right before the statement.
"""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "ma57_amd" / "csrc"


def _statements(src):
    for m in re.finditer(r"\basm(?:\s+volatile)?\s*\(", src):
        depth, end = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(src[end], 0)
            end += 1
        yield src[m.end():end]


@pytest.mark.parametrize("name", ["factor_kernels.hip", "solve_kernels.hip", "cb_syrk.hip"])
def test_dpp_reads_follow_their_wait_states(name):
    src = re.sub(r"//[^\n]*", "", (CSRC / name).read_text())
    macros = [m for m, body in re.findall(r"#define (\w+)\([^)]*\)([^\n]*)", src) if "_dpp" in body]
    reads = re.compile("|".join(["_dpp"] + [rf"\b{m}\(" for m in macros]))
    for s in _statements(src):
        if reads.search(s):
            assert re.match(r'\s*"s_nop [1-9]', s), s[:120]
