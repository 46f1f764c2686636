"""Assembly tiles: parent fronts around the tile sizes (64, 128 and 256 rows), children that meet them in runs.

Independent leaf blocks, each coupled to its own random rows of a dense separator: the separator's front sums A and
every leaf's contribution block.  Tolerances: a small multiple of n * unit roundoff
with a growth factor of 100 in the backward error; the counts of eigenvalue signs are exact.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from ma57_amd import problems as P
from ma57_amd.solver import SymLDLT, OrderingType, Precision

from test_gpu_parity import _lapack_inertia

pytestmark = pytest.mark.gpu


def _leaves_and_separator(nsep, leaves, leaf, seed):
    rng = np.random.default_rng(seed)
    n = leaves * leaf + nsep
    A = np.zeros((n, n))
    s0 = leaves * leaf
    R = rng.standard_normal((nsep, nsep))
    A[s0:, s0:] = (R + R.T) / 2
    for k in range(leaves):
        o = k * leaf
        R = rng.standard_normal((leaf, leaf))
        A[o:o + leaf, o:o + leaf] = (R + R.T) / 2 + leaf * np.eye(leaf) * (1 if k % 2 else -1)
        rows = s0 + rng.choice(nsep, size=max(1, (nsep * (k + 1)) // (leaves + 1)), replace=False)
        A[np.ix_(rows, np.arange(o, o + leaf))] = rng.standard_normal((rows.size, leaf))
        A[np.ix_(np.arange(o, o + leaf), rows)] = A[np.ix_(rows, np.arange(o, o + leaf))].T
    return A


@pytest.mark.parametrize("prec,eps", [(Precision.FP64, 2.0 ** -53), (Precision.FP32, 2.0 ** -24)])
@pytest.mark.parametrize("nsep", [1, 17, 63, 64, 65, 127, 128, 129, 255, 257, 300, 530])
def test_children_add_into_parent_tiles(nsep, prec, eps):
    A = _leaves_and_separator(nsep, 7, 12, nsep)
    n = A.shape[0]
    L = sp.csc_matrix(np.tril(A))
    for tile in (64, 32, 16):
        s = SymLDLT()
        s.setOrdering(OrderingType.AMD)
        s.setPrecision(prec)
        s.analyzePattern(L)
        s.setTuning(64, tile, True)
        s.factorize(L)
        i = s.inertia()
        if prec == Precision.FP64:
            assert (i.n_pos, i.n_neg, i.n_zero) == (*_lapack_inertia(A), 0)
        b = np.random.default_rng(n).standard_normal((n, 3))
        assert P.backward_error(L, s.solve(b), b) <= 100 * n * eps
