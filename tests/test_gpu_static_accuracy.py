"""Static pivots without any perturbation on random fronts: the multipliers are unbounded, the factors still exact
for a matrix close to A entry by entry.

A = L D L^T up to roundings of its own terms: entry (i, j) is a sum of at most n products l_iq d_q l_jq, each rounded
a few times, so against |L| |D| |L|^T it is off by about sqrt(n) u for independent roundings; twice that is allowed.
A substitution by explicit inverses, or multipliers that differ from the ones used in the products, is not: errors of
up to 1600 u at 300 rows.
"""
import numpy as np
import pytest

from ma57_amd.solver import dense_factor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n,ne", [(193, 193), (250, 250), (300, 300), (300, 249), (330, 65), (400, 400)])
def test_componentwise_backward_error(n, ne, exact):
    for seed in range(6):
        R = np.random.default_rng(1000 * n + seed).standard_normal((n, n))
        A = (R + R.T) / 2
        g = dense_factor(A, n_eligible=ne, static_mode=True, static_delta=1e-300, static_rel_floor=1e-300,
                         exact_panel=exact)
        assert g["n_factored"] == ne and g["num_perturbed"] == 0
        L = np.tril(g["A"], -1)[:, :ne].astype(np.longdouble)
        L[np.arange(ne), np.arange(ne)] = 1
        D = g["d_diag"][:ne].astype(np.longdouble)
        E = np.abs((L * D) @ L[:ne].T - A[:, :ne]) / ((np.abs(L) * np.abs(D)) @ np.abs(L[:ne]).T)
        assert np.tril(E).max() <= 2 * np.sqrt(n) * 2.0 ** -53, (seed, float(np.tril(E).max() * 2.0 ** 53))
