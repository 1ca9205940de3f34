"""The inverse from the tile factor at the sizes where the sweep's blocks
change: with the transposed copy up to 2,560 rows in two launches a column,
beyond (and without it) in blocked stages of 96 x 96 blocks for tiles of a
multiple of 192 and 64 x 64 blocks else; one tile, ragged last tiles, tiles
whose 64-row blocks straddle the 96-row ones."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
KN = "univariate_matern_nuggets_stationary"
SIZES = [(60, 64), (321, 64), (900, 64), (700, 128), (193, 192), (900, 192), (1500, 576), (1281, 320), (2560, 64),
         (2100, 128), (2200, 192), (2600, 64), (2600, 128), (2600, 192), (2100, 960)]


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


@pytest.mark.parametrize("n,ts", SIZES)
def test_inverse(lib, n, ts):
    """Without the transposed copy: max |Z - S^-1| <= 8 (n + 64) eps cond(S)
    max |S^-1| (backward error (n + 1) eps of the factor, 64 eps of the products
    with block inverses, c = 8); the diagonal tiles are symmetric."""
    x, y = lib.generate_xy_loc(n, 7)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg((1.0, 0.1, 0.5), x, y)
    S = np.tril(M.to_numpy())
    S = S + np.tril(S, -1).T + 0.1 * np.eye(n)
    M.from_numpy(S)
    assert M.potrf() == 0
    M.potri()
    Z = M.to_numpy()
    M.close()
    for k in range(0, n, ts):
        assert np.array_equal(Z[k:k + ts, k:k + ts], Z[k:k + ts, k:k + ts].T)
    ref = np.linalg.inv(S)
    tol = 8 * (n + 64) * EPS * np.linalg.cond(S) * np.max(np.abs(ref))
    assert np.max(np.abs(np.tril(Z - ref))) <= tol


@pytest.mark.parametrize("n,ts", SIZES)
def test_trace(lib, n, ts):
    """With it, through the gradient: sigma^2 l_sigma^2 + tau^2 l_tau^2 =
    (z^T S^-1 z - tr(S^-1 S)) / 2 with tr = n, to the same relative error."""
    x, y = lib.generate_xy_loc(n, 7)
    th = np.array([1.2, 0.1, 0.5, 0.3])
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg(th[:3], x, y)
    S = np.tril(M.to_numpy())
    M.close()
    S = S + np.tril(S, -1).T + th[3] * np.eye(n)
    z = np.random.default_rng(n).standard_normal(n)
    m = lib.ExactMLE(x, y, ts, kernel=KN)
    m.set_z(z)
    _, g = m.loglik(th, grad=True)
    m.close()
    q = z @ np.linalg.solve(S, z)
    tol = 8 * (n + 64) * EPS * np.linalg.cond(S) * (q + n)
    assert abs(th[0] * g[0] + th[3] * g[3] - 0.5 * (q - n)) <= tol
