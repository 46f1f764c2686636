"""The static pivot rule on diagonal matrices, whose pivots are their entries: LDS fronts, exact and speculative panels.

A pivot below the floor in its expected direction moves by delta times its expected sign; any integer is accepted as
a sign.  NaN and infinite pivots are taken as they are and are no perturbation.
"""
import numpy as np
import pytest

from ma57_amd.solver import dense_factor

pytestmark = pytest.mark.gpu

DELTA, FLOOR = 1e-4, 1e-4


def _rule(d, sign, floor):
    towards = d if sign > 0 else -d if sign < 0 else np.abs(d)
    s = sign if sign else np.where(d >= 0, 1.0, -1.0)
    return np.where(towards < floor, d + s * DELTA, d)


@pytest.mark.parametrize("n,exact", [(40, True), (200, True), (200, False), (700, False)])
@pytest.mark.parametrize("sign", [-3, -1, 0, 1, 2])
def test_rule_for_any_sign(n, exact, sign):
    d = np.linspace(-1e-3, 1e-3, n)
    d[0] = 1.0  # the floor is FLOOR times the largest entry
    g = dense_factor(np.diag(d), static_mode=True, static_delta=DELTA, static_rel_floor=FLOOR, exact_panel=exact,
                     expected_sign=np.full(n, sign))
    want = _rule(d, sign, FLOOR)
    # (d + s delta in one rounding or two)
    assert np.allclose(g["d_diag"], want, rtol=2.0 ** -52, atol=DELTA * 2.0 ** -50)
    assert g["num_perturbed"] == (want != d).sum()
    # a sum of at most n terms, each within an ulp of an entry
    assert g["total_perturbation"] == pytest.approx(np.abs(want - d).sum(), rel=n * 2.0 ** -50)
    assert g["inertia"] == ((want > 0).sum(), (want < 0).sum(), 0)


@pytest.mark.parametrize("n", [40, 200])
@pytest.mark.parametrize("last", [np.nan, np.inf, -np.inf])
def test_non_finite_pivot_is_no_perturbation(n, last):
    d = np.linspace(-1e-3, 1e-3, n)
    d[0], d[-1] = 1.0, last
    g = dense_factor(np.diag(d), static_mode=True, static_delta=DELTA, static_rel_floor=FLOOR)
    want = _rule(d, 0, FLOOR if np.isnan(last) else np.inf)  # the floor follows the largest entry that is a number
    if np.isinf(last):
        want[-1] = last
    assert np.allclose(g["d_diag"], want, rtol=2.0 ** -52, atol=DELTA * 2.0 ** -50, equal_nan=True)
    changed = int((want[:-1] != d[:-1]).sum())
    assert g["num_perturbed"] == changed
    assert g["total_perturbation"] == pytest.approx(np.abs(want[:-1] - d[:-1]).sum(), rel=n * 2.0 ** -50)
