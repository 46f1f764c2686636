"""The last pass of the speculative panel step: its workgroups run in any order.

Workgroup 0 of a front advances the front's state in the same launch in which the others restore their rows after a
failed test, and nothing orders them.  A workgroup that read a word workgroup 0 writes would restore rows of another
panel.  Which words that is shows in the kernel's source, on the CPU; the GPU case factors many fronts whose panels
all fail a test.
"""
import re
from pathlib import Path

import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision

SOURCE = Path(__file__).resolve().parent.parent / "ma57_amd" / "csrc" / "factor_kernels.hip"


def _kernel(name):
    src = re.sub(r"//[^\n]*", "", SOURCE.read_text())
    at = src.index("{", src.index(f" {name}(const int* list"))
    depth, end = 1, at + 1
    while depth:
        depth += {"{": 1, "}": -1}.get(src[end], 0)
        end += 1
    return src[at:end]


def test_what_every_workgroup_reads_no_workgroup_writes():
    body = _kernel("k_spec_apply")
    everyone, lead = body.split("if (w != 0) return;")
    assign = r"\b(fd\.\w+\[[^\]]*\]|\*rec\.\w+|rec\.(?!colmax)\w+\[[^\]]*\])\s*[+\-*/|&^]?=(?!=)"
    word = r"\b(?:fd|rec)\.(\w+)"
    written = {re.search(word, m).group(1) for m in re.findall(assign, body)}
    written |= set(re.findall(r"atomic\w+\(fd\.(\w+)", body))
    assert {"kcur", "nF", "pcount", "cbDone", "inertia"} <= written
    read = set(re.findall(word, re.sub(assign, "", everyone)))
    assert {"m", "nE", "F", "origMaxBits"} <= read
    assert not read & written
    # the column maxima have two buffers: this panel's is read, the next one's cleared
    buffers = r"rec\.colmax\[([^\]]*) \* P"
    assert re.findall(buffers, everyone) == ["parity"] and re.findall(buffers, lead) == ["(parity ^ 1)"]


@pytest.mark.gpu
@pytest.mark.parametrize("prec,eps", [(Precision.FP64, 2.0 ** -53), (Precision.FP32, 2.0 ** -24)])
def test_many_fronts_with_failing_panels(prec, eps):
    """64 independent fronts of 330 rows, a planted 2x2 pivot in every panel (tolerance: a small multiple of
    n * unit roundoff with a growth factor of 100 in the backward error)."""
    rng = np.random.default_rng(12)
    n, blocks = 330, []
    for _ in range(64):
        R = rng.standard_normal((n, n)) / np.sqrt(n)
        A = (R + R.T) / 2 + np.diag(np.where(rng.random(n) < 0.5, -1.0, 1.0) * rng.uniform(2.0, 4.0, n))
        for c in range(int(rng.integers(1, 50)), n - 1, 50):
            A[c, c] = A[c + 1, c + 1] = 0.0
            A[c, c + 1] = A[c + 1, c] = 3.0
        blocks.append(A)
    ev = np.concatenate([np.linalg.eigvalsh(A) for A in blocks])
    L = sp.csc_matrix(sp.tril(sp.block_diag(blocks)))
    s = SymLDLT()
    s.setOrdering(OrderingType.AMD)
    s.setPrecision(prec)
    s.analyzePattern(L)
    s.setTuning(64, 64, True, 0)
    b = rng.standard_normal((64 * n, 2))
    for _ in range(4):
        s.factorize(L)
        i = s.inertia()
        assert (i.n_pos, i.n_neg, i.n_zero) == (int((ev > 0).sum()), int((ev < 0).sum()), 0)
        assert P.backward_error(L, s.solve(b), b) <= 100 * n * eps
