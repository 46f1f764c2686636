"""Parents with more than 64 children (they are looked at 64 at a time), and own rows whose ancestors' rows are split.

Tolerances: a small multiple of n * unit roundoff with a growth factor of 100 in the backward error.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision

pytestmark = pytest.mark.gpu

PRECISIONS = [(Precision.FP64, 2.0 ** -53), (Precision.FP32, 2.0 ** -24)]


def _bordered(nsep, leaves, leaf, rows, seed):
    """Independent leaves, each coupled to `rows` random rows of a dense separator."""
    rng = np.random.default_rng(seed)
    s0 = leaves * leaf
    A = sp.lil_matrix((s0 + nsep, s0 + nsep))
    R = rng.standard_normal((nsep, nsep))
    A[s0:, s0:] = np.tril(R + R.T) / 2
    for k in range(leaves):
        o = k * leaf
        R = rng.standard_normal((leaf, leaf))
        A[o:o + leaf, o:o + leaf] = np.tril((R + R.T) / 2 + leaf * np.eye(leaf) * (1 if k % 2 else -1))
        at = s0 + np.sort(rng.choice(nsep, size=rows, replace=False))
        for j in range(o, o + leaf):
            A[at, j] = rng.standard_normal((rows, 1))
    return A.tocsc()


def _solver(L, prec):
    s = SymLDLT()
    s.setOrdering(OrderingType.Natural)
    s.setPrecision(prec)
    s.analyzePattern(L)
    s.factorize(L)
    return s


@pytest.mark.parametrize("prec,eps", PRECISIONS)
@pytest.mark.parametrize("leaves", [63, 64, 65, 128, 129, 200])
def test_children_in_groups(leaves, prec, eps):
    L = _bordered(90, leaves, 5, 40, leaves)
    s = _solver(L, prec)
    sn = s.symbolicFactor().supernodes
    assert len(sn) > leaves  # the separator's front has every leaf below it
    b = np.random.default_rng(leaves).standard_normal((L.shape[0], 3))
    assert P.backward_error(L, s.solve(b), b) <= 100 * L.shape[0] * eps


@pytest.mark.parametrize("prec,eps", PRECISIONS)
@pytest.mark.parametrize("leaf,nsep", [(70, 513), (70, 1500), (190, 1100), (100, 2600)])
def test_split_ancestor_rows(leaf, nsep, prec, eps):
    """Leaves of 3 to 6 own blocks with more than 512 rows below them: the backward product runs in chunks of rows
    whose partial sums the own-row kernel adds up (four chunks at a time)."""
    L = _bordered(nsep, 3, leaf, nsep, leaf + nsep)
    s = _solver(L, prec)
    n = L.shape[0]
    for nrhs in (1, 16, 17, 65):
        b = np.random.default_rng(n + nrhs).standard_normal((n, nrhs))
        assert P.backward_error(L, s.solve(b), b) <= 100 * n * eps
