"""The panel kernel and the multipliers of the rows below it, pivot by pivot path.

Random indefinite fronts need 2x2 pivots and interchanges in most blocks of 16 columns.  Sizes lie around the
kernel's own edges: rows held in LDS, in registers (128, 256, 512, 1024 and 2048 rows) and streamed, fronts whose
rows are all held by the panel (at most 256), panels and blocks with a remainder, a 2x2 pivot across a panel's end.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision, dense_factor

from test_gpu_parity import _lapack_inertia, _reconstruct

pytestmark = pytest.mark.gpu


def _indefinite(n, seed):
    R = np.random.default_rng(seed).standard_normal((n, n))
    return (R + R.T) / 2.0


@pytest.mark.parametrize("n,ne", [(193, 193), (256, 200), (257, 257), (300, 17), (400, 65), (512, 512), (513, 449),
                                  (1025, 1000), (1100, 1100), (2049, 2047), (2113, 2113)])
def test_exact_panel_factors_random_fronts(n, ne):
    A = _indefinite(n, n + ne)
    g = dense_factor(A, n_eligible=ne, exact_panel=True)
    assert g["n_factored"] == ne
    assert any(k == 2 for _, k in g["pivots"])
    A11 = A[:ne, :ne]
    assert g["inertia"] == (*_lapack_inertia(A11), 0)
    p = g["perm"][:ne]
    assert np.linalg.norm(_reconstruct(g, ne) - A11[np.ix_(p, p)]) / np.linalg.norm(A11) < 1e-10
    if ne < n:
        S = A[ne:, ne:] - A[ne:, :ne] @ np.linalg.solve(A11, A[:ne, ne:])
        assert np.abs(np.tril(g["A"][ne:, ne:]) - np.tril(S)).max() <= 1e-8 * max(1.0, np.abs(S).max())


@pytest.mark.parametrize("n", [100, 257, 520, 1030])
def test_fp32_panels_refine(n):
    A = _indefinite(n, n)
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
