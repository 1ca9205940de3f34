"""The gradient's table (x^nu (x K_{nu+1} - 2 nu K_nu) and dM/dnu) where it can
go wrong: the ends of its range (2^-20 and 130, beyond which entries are
evaluated directly), interval boundaries on both grids and their change at
x = 2, for small, half-integer, integer and larger orders."""
from __future__ import annotations

import numpy as np
import pytest
from scipy.special import digamma, gammaln

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
EDGES = np.concatenate([
    2.0 ** -20 * np.array([0.25, 1 - 1e-15, 1.0, 1 + 1e-15, 1.5]),
    [1.0, 1.0625, 1.9375, 2.0, 2.0625, 3.0, 17.5, 129.9375, 130.0, 131.0, 400.0],
])


def _functions(x, nu):
    """B = c x^nu (x K_{nu+1} - 2 nu K_nu), V = d(c x^nu K_nu)/dnu and the sums
    of the magnitudes of their terms, from the integrals of K over cosh in
    extended precision."""
    L = np.longdouble
    h = L(0.04)
    x, nu = L(x), L(nu)
    t = h * np.arange(int(np.arccosh(12000.0 / float(x)) / float(h)) + 2)
    w = np.where(t == 0, L(0.5), L(1.0)) * h * np.exp(-x * (np.cosh(t) - 1))
    f = np.exp(nu * np.log(x) - x) / L(2.0) ** (nu - 1) / np.exp(L(gammaln(float(nu))))
    K, K1, Km = (f * np.sum(w * np.cosh(o * t)) for o in (nu, nu + 1, nu - 1))
    dK = f * np.sum(w * t * np.sinh(nu * t))
    dc = -np.log(L(2.0)) - L(digamma(float(nu)))
    return x * Km, x * K1 + 2 * nu * K, (dc + np.log(x)) * K + dK, (abs(dc) + abs(np.log(x))) * K + dK


@pytest.mark.parametrize("nu", [0.05, 0.5, 0.8, 1.0, 1.37, 3.2])
def test_derivatives_at_the_edges(nu):
    """Two locations at distance x, unit range, variance and nugget, z = (3, 3):
    the gradient is -w B and -w V with w = (C^-1)_12 - alpha_1 alpha_2, both
    terms negative.  Errors to (4,000 + 8 x + 8 nu |log x| + 8 |log Gamma(nu)|)
    eps of the terms' magnitudes: rounded arguments of exponentials and powers,
    and a few thousand roundings of a series with its derivative."""
    import exageostat_amd as lib
    rng = np.random.default_rng(2)
    xs = np.unique(np.concatenate([EDGES, np.nextafter(EDGES, 0.0), np.nextafter(EDGES, 1e9),
                                   np.exp(rng.uniform(np.log(1e-7), np.log(200.0), 60))]))
    m = lib.ExactMLE(np.array([0.0, 1.0]), np.zeros(2), 64, kernel="univariate_matern_nuggets_stationary")
    m.set_z(np.array([3.0, 3.0]))
    worst = 0.0
    for x in xs:
        m.x[1] = x
        ll, g = m.loglik((1.0, 1.0, nu, 1.0), grad=True)
        B, magB, V, magV = _functions(x, nu)
        M = (magB - B) / (4 * np.longdouble(nu))  # x K_{nu+1} - x K_{nu-1} = 2 nu K_nu
        w = -M / (4 - M * M) - 9 / (2 + M) ** 2
        tol = (4000 + 8 * x + 8 * nu * abs(np.log(x)) + 8 * abs(gammaln(nu))) * EPS
        worst = max(worst, abs(g[1] / -w - B) / (tol * magB), abs(g[2] / -w - V) / (tol * magV))
    m.close()
    assert worst <= 1.0, float(worst)
