"""Tile steps of the FP64 factorisation (tile-column panels, trailing updates
with one and with two panels) at every block shape of the update and with few
64-column blocks per tile column: 211 block columns, so that they run before
the last 200 go into one launch."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
N = 13500


@pytest.mark.parametrize("ts", [64, 320, 448,  # 64 x 64 blocks
                                128, 256, 512,  # 128 x 128
                                192, 576])  # 96 x 192
def test_factor(ts):
    """L L^T v against S v for a vector of signs: |error| <= 8 (n + 64) eps per
    entry of S (the factor's residual), sqrt(n) of them at random signs, and
    five standard deviations."""
    import exageostat_amd as lib
    x, y = lib.generate_xy_loc(N, 3)
    M = lib.DeviceMatrix(N, N, ts, lower=True)
    M.dcmg((1.0, 0.1, 0.5), x, y)
    S = np.tril(M.to_numpy())
    assert M.potrf() == 0
    L = M.to_numpy()
    M.close()
    v = np.where(np.random.default_rng(0).random(N) < 0.5, -1.0, 1.0)
    Sv = S @ v + S.T @ v - np.diag(S) * v
    assert np.max(np.abs(L @ (L.T @ v) - Sv)) <= 5 * np.sqrt(N) * 8 * (N + 64) * EPS
    assert np.all(L[:64, 64:] == 0.0) and np.all(L[-64:-1, -1] == 0.0)
