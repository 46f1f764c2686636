"""Panels of fronts with more than 512 rows: where blocks of columns keep few of theirs, columns are taken one by one.

Stretches of columns that pass the first pivot test, of columns that fail it, and mixtures, around the register
variants' limits (1,024 and 2,048 rows) and streamed.  Inertia against LAPACK; reconstruction and refined backward
error as for the other panel tests.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision, dense_factor

from test_gpu_parity import _lapack_inertia, _reconstruct

pytestmark = pytest.mark.gpu


def _mixture(n, stretch):
    """Dominant rows, every other stretch of them replaced by planted 2x2 pivots with zero diagonals."""
    rng = np.random.default_rng(n + stretch)
    R = rng.standard_normal((n, n)) / np.sqrt(n)
    A = (R + R.T) / 2 + np.diag(np.where(rng.random(n) < 0.5, -1.0, 1.0) * rng.uniform(2.0, 4.0, n))
    for c in range(0, n - 1, 2):
        if (c // stretch) % 2 == 0:
            A[c, c] = A[c + 1, c + 1] = 0.0
            A[c, c + 1] = A[c + 1, c] = 3.0
    return A


@pytest.mark.parametrize("n,ne", [(513, 513), (700, 650), (1024, 1024), (1025, 1025), (1500, 1400), (2100, 2100)])
@pytest.mark.parametrize("stretch", [2, 6, 10, 40])
def test_runs_of_failing_columns(n, ne, stretch):
    A = _mixture(n, stretch)
    g = dense_factor(A, n_eligible=ne, exact_panel=True)
    assert g["n_factored"] == ne
    assert any(k == 2 for _, k in g["pivots"])
    A11 = A[:ne, :ne]
    assert g["inertia"] == (*_lapack_inertia(A11), 0)
    p = g["perm"][:ne]
    assert np.linalg.norm(_reconstruct(g, ne) - A11[np.ix_(p, p)]) / np.linalg.norm(A11) < 1e-10


@pytest.mark.parametrize("n", [600, 1100, 2100])
def test_fp32_fronts_refine(n):
    R = np.random.default_rng(n).standard_normal((n, n))
    A = (R + R.T) / 2
    L = sp.csc_matrix(np.tril(A))
    s = SymLDLT()
    s.setOrdering(OrderingType.AMD)
    s.setPrecision(Precision.FP32)
    s.analyzePattern(L)
    s.setTuning(64, 32, False)
    s.factorize(L)
    i = s.inertia()
    assert (i.n_pos, i.n_neg, i.n_zero) == (*_lapack_inertia(A), 0)
    b = np.random.default_rng(n + 1).standard_normal((n, 2))
    assert P.backward_error(L, s.solveWithRefinement(L, b).x, b) <= 1e-12
