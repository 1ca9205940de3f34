"""Triangular solves in one launch, L x = b and L^T x = b, by their residuals
at the sizes where the strips of a tile change: one block per tile, one part
(2 to 4 blocks), parts that are not full (5, 6, 9, 13 blocks), four full parts
(16 blocks), one tile, and ragged last tiles."""
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


@pytest.mark.parametrize("n,ts", [(1, 64), (64, 64), (1000, 64), (129, 128), (700, 192), (1300, 256), (961, 320),
                                  (1537, 384), (1200, 576), (2500, 832), (900, 960), (3100, 1024)])
def test_residual(lib, n, ts):
    """|L x - b| row by row.  The sums over the other tiles and the partials
    have fewer than n + 64 terms each: (n + 64) eps |L| |x|.  The diagonal
    tile L_d is applied through its inverse X, which is off by at most
    c ts eps |X| |L_d| |X| (c = 8): L_d (X w) is off from w = L_d x by
    8 ts eps |L_d| |X| |L_d| |X| |w|."""
    x, y = lib.generate_xy_loc(n, 5)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg((1.0, 0.1, 0.5), x, y)
    assert M.potrf() == 0
    b = np.random.default_rng(n).standard_normal(n)
    got = [M.trsv(b), M.trsv(b, trans=True)]
    again = [M.trsv(b), M.trsv(b, trans=True)]
    L = M.to_numpy()
    M.close()
    for A, v, v2 in zip((L, L.T), got, again):
        assert np.array_equal(v, v2)
        bound = (n + 64) * EPS * (np.abs(A) @ np.abs(v))
        for k in range(0, n, ts):
            D = A[k:k + ts, k:k + ts]
            X = np.abs(np.linalg.inv(D))
            w = np.abs(D @ v[k:k + ts])
            D = np.abs(D)
            bound[k:k + ts] += 8 * ts * EPS * (D @ (X @ (D @ (X @ w))))
        assert np.all(np.abs(A @ v - b) <= bound)
