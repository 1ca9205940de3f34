"""The correlation table of covariance generation at the places where it can
go wrong: the ends of its range (2^-20 and 130, beyond which entries are
evaluated directly), interval boundaries on both grids and their change at
x = 2, smoothness near integers, small and large, and orders whose K_nu
overflows inside the range."""
from __future__ import annotations

import numpy as np
import pytest
from scipy.special import gammaln, kv

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
EDGES = np.concatenate([
    2.0 ** -20 * np.array([0.25, 1 - 1e-15, 1.0, 1 + 1e-15, 1.5]),
    [1.0, 1.0625, 1.9375, 2.0, 2.0625, 3.0, 17.5, 129.9375, 130.0, 131.0, 400.0],
])


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


def _matern(x, nu):
    """K_nu from its integral over cosh in extended precision (the trapezoidal
    rule converges exponentially); scipy's kv is up to 9e-14 off here."""
    x = x.astype(np.longdouble)
    h = np.longdouble(0.04)
    t = h * np.arange(int(np.arccosh(12000.0 / float(x.min())) / float(h)) + 2)
    w = np.where(t == 0, 0.5, 1.0) * h * np.cosh(np.longdouble(nu) * t)
    k = np.array([np.sum(w * np.exp(-xi * (np.cosh(t) - 1))) for xi in x])
    return (np.exp(np.longdouble(nu) * np.log(x) - x) * k / np.longdouble(2.0) ** (nu - 1) /
            np.exp(np.longdouble(gammaln(nu))))


@pytest.mark.parametrize("nu", [0.05, 0.499, 0.55, 1.0, 1.0 + 1e-9, 1.37, 3.2, 12.3])
def test_correlations_at_the_edges(lib, nu):
    """Relative error at most (200 + 4 x + 4 nu |log x| + 4 |log Gamma(nu)|)
    eps: the exponentials' and powers' arguments are rounded, the rest is some
    hundred roundings."""
    rng = np.random.default_rng(1)
    x = np.unique(np.concatenate([EDGES, np.nextafter(EDGES, 0.0), np.nextafter(EDGES, 1e9),
                                  np.exp(rng.uniform(np.log(1e-7), np.log(200.0), 900))]))
    n = len(x)
    M = lib.DeviceMatrix(1, n, 64, lower=False)
    M.dcmg((1.0, 1.0, nu), np.zeros(1), np.zeros(1), x, np.zeros(n))
    got = M.to_numpy()[0]
    M.close()
    ref = _matern(x, nu)
    tol = (200 + 4 * x + 4 * nu * np.abs(np.log(x)) + 4 * abs(gammaln(nu))) * EPS
    assert np.all(np.abs(got - ref) <= tol * ref), (np.abs(got - ref) / (tol * ref)).max()


def test_order_that_overflows(lib):
    """K_60 overflows below x = 2.9e-4: those entries come out as the direct
    evaluation gives them, their finite neighbours in the same interval are
    not affected."""
    nu = 60.0
    x = np.exp(np.linspace(np.log(1e-4), np.log(1e-2), 400))
    M = lib.DeviceMatrix(1, len(x), 64, lower=False)
    M.dcmg((1.0, 1.0, nu), np.zeros(1), np.zeros(1), x, np.zeros(len(x)))
    got = M.to_numpy()[0]
    M.close()
    fine = np.isfinite(kv(nu + 1.0, x))
    assert fine.any() and not fine.all()
    # M = 1 - x^2 / (4 (nu - 1)) + ..., and the factors' arguments are rounded
    tol = (200 + 4 * nu * np.abs(np.log(x)) + 4 * gammaln(nu)) * EPS
    assert np.all(np.abs(got[fine] - (1.0 - x[fine] ** 2 / (4 * (nu - 1)))) <= tol[fine] + x[fine] ** 4)
