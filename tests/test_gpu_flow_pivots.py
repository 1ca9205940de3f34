"""Pivots outside the range of the factorisation's fast reciprocals and roots:
infinite ones (a row whose variance has no bound: its column of L is zero and
the rows after it do not see it), subnormal ones and the ends of the normal
range, at the edges of the 16-column panels and the 64-column blocks."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


def _matrix(lib, n, ts):
    x, y = lib.generate_xy_loc(n, 3)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg((1.0, 0.1, 0.5), x, y)
    S = np.tril(M.to_numpy())
    return M, S + np.tril(S, -1).T


@pytest.mark.parametrize("n,ts,at", [(200, 64, 0), (200, 64, 5), (200, 64, 15), (200, 64, 16), (200, 64, 63),
                                     (200, 64, 64), (200, 128, 100), (200, 64, 199), (1, 64, 0)])
def test_infinite_pivot(lib, n, ts, at):
    """Against the factor with 2^600 in its place, whose column below it is
    under 2^-300 and whose other rows are the same: entries to 64 (n + 64) eps:
    the residual's bound of 8 (n + 64) eps, times a condition number of the
    leading rows below 8."""
    M, S = _matrix(lib, n, ts)
    S[at, at] = 2.0 ** 600
    ref = np.linalg.cholesky(S)
    ref[at, at] = np.inf
    ref[at + 1:, at] = 0.0
    S[at, at] = np.inf
    M.from_numpy(S)
    assert M.potrf() == 0
    L = M.to_numpy()
    b = np.cos(np.arange(n))
    y = M.trsv(b)
    M.close()
    assert L[at, at] == np.inf and np.all(L[at + 1:, at] == 0.0)
    rest = np.delete(np.arange(n), at)
    assert np.all(np.isfinite(L[rest])) and y[at] == 0.0 and np.all(np.isfinite(y))
    fin = np.isfinite(ref)
    assert np.max(np.abs(L[fin] - ref[fin]), initial=0.0) <= 64 * (n + 64) * EPS


@pytest.mark.parametrize("value", [5e-324, 3e-310, 2.3e-308, 1e-302, 1e302, 1.7e308])
@pytest.mark.parametrize("at", [0, 17, 63, 70, 199])
def test_extreme_pivot(lib, value, at):
    """Alone in its row and column: its root (two roundings), and the factor
    of the other rows as with 1 in its place, to 8 (n + 64) eps."""
    n, ts = 200, 64
    M, S = _matrix(lib, n, ts)
    S[at, :] = S[:, at] = 0.0
    S[at, at] = 1.0
    M.from_numpy(S)
    assert M.potrf() == 0
    ref = M.to_numpy()
    S[at, at] = value
    M.from_numpy(S)
    assert M.potrf() == 0
    L = M.to_numpy()
    M.close()
    assert abs(L[at, at] - np.sqrt(value)) <= 2 * EPS * np.sqrt(value)
    L[at, at] = ref[at, at]
    assert np.max(np.abs(L - ref)) <= 8 * (n + 64) * EPS


def test_negative_pivot_after_an_extreme_one(lib):
    """The first failing column is still the one reported."""
    n, ts = 200, 64
    M, S = _matrix(lib, n, ts)
    S[20, 20] = np.inf
    S[25, 25] = -1.0
    M.from_numpy(S)
    assert M.potrf() == 26
    S[20, 20] = -1.0
    S[25, 25] = np.inf
    M.from_numpy(S)
    assert M.potrf() == 21
    M.close()
