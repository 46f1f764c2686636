"""Every solve kernel whose work is sized by the plan notices a front that has outgrown it.

No layout rule lets that happen, so the guard is looked at in the source: the kernel compares the front's pivots with
what was planned for it and raises the error word instead of leaving products out.
"""
import re
from pathlib import Path

import pytest

SOURCE = Path(__file__).resolve().parent.parent / "ma57_amd" / "csrc" / "solve_kernels.hip"


@pytest.mark.parametrize("kernel", ["k_fwd_own", "k_bwd_own", "k_fwd_chain", "k_bwd_chain", "k_fwd_delta", "k_bwd_anc"])
def test_kernel_raises_when_a_front_outgrew_its_plan(kernel):
    src = re.sub(r"//[^\n]*", "", SOURCE.read_text())
    body = re.search(rf"__global__[^{{;]*?\b{kernel}\(.*?\n}}\n", src, re.S).group(0)
    assert re.search(r"\bint\s*\*\s*err\b", body.split("{")[0])
    assert re.search(r"if \([^;]*(nOwn|nD) > [^;]*raiseError\(err, 2\);", body, re.S)
