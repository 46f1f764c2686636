"""Own rows of short chains: blocks of 32 rows around the limits, right-hand sides around groups of 16.

Dense indefinite fronts (2x2 pivots in most blocks, so also across 32-row boundaries) of one to seven own blocks;
the largest goes to the chain kernels.  Backward error: FP64 factors with threshold pivoting give a small multiple
of n * 2^-53, FP32 ones n * 2^-24; both get a growth factor of 100.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,eps", [(Precision.FP64, 2.0 ** -53), (Precision.FP32, 2.0 ** -24)])
@pytest.mark.parametrize("n", [65, 96, 97, 128, 129, 191, 192, 193, 224])
def test_own_rows_solve(n, prec, eps):
    R = np.random.default_rng(n).standard_normal((n, n))
    L = sp.csc_matrix(np.tril((R + R.T) / 2.0))
    s = SymLDLT()
    s.setOrdering(OrderingType.AMD)
    s.setPrecision(prec)
    s.analyzePattern(L)
    s.setTuning(64, 32, False)
    s.factorize(L)
    for nrhs in (1, 15, 16, 17, 64, 65):
        b = np.random.default_rng(n + nrhs).standard_normal((n, nrhs))
        assert P.backward_error(L, s.solve(b), b) <= 100 * n * eps
