"""Matrices with one NaN or infinite entry: what the reference takes is taken, and a program sees no error.

NaN compares as below nothing, so pivots are accepted past it as in the reference; the oracle says how many.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd.solver import SymLDLT, OrderingType, dense_factor

pytestmark = pytest.mark.gpu


def _matrix(n, dominant):
    R = np.random.default_rng(n).standard_normal((n, n))
    A = (R + R.T) / 2
    if dominant:
        A += np.diag(np.where(np.arange(n) % 2, 1.0, -1.0)) * 3 * n
    return A


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("dominant", [True, False])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n", [40, 200, 300])
def test_pivots_taken(n, value, dominant, exact, oracle):
    for i, j in ((0, 0), (20, 20), (25, 22), (n - 1, 3), (n - 1, n - 1)):
        A = _matrix(n, dominant)
        A[i, j] = A[j, i] = value
        assert dense_factor(A, exact_panel=exact)["n_factored"] == oracle.dense_factor(A)["n_factored"], (i, j)
    for i in (0, 20, n - 1):  # a column of its own
        A = _matrix(n, dominant)
        A[i, :] = A[:, i] = 0.0
        A[i, i] = value
        assert dense_factor(A, exact_panel=exact)["n_factored"] == oracle.dense_factor(A)["n_factored"], i


@pytest.mark.parametrize("speculative", [True, False])
@pytest.mark.parametrize("n", [40, 200, 300])
def test_nan_reaches_the_solution(n, speculative):
    A = _matrix(n, True)
    pattern = sp.csc_matrix(np.tril(A))
    s = SymLDLT()
    s.setOrdering(OrderingType.AMD)
    s.analyzePattern(pattern)
    s.setTuning(64, 64, speculative, 0)
    A[n - 1, 3] = np.nan
    L = pattern.copy()
    L.data[:] = np.concatenate([A[j:, j] for j in range(n)])
    s.factorize(L)
    assert np.isnan(s.solve(np.ones(n))).any()
