"""Dataflow Cholesky against the matrix it factors, at the sizes where its
block and task ranges change: one block, ragged last blocks, row groups that
are not full, tile columns with few blocks, the last padded blocks, and the
sizes around the switch from the tile steps to one launch (200 block
columns)."""
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


def _factor(lib, n, ts, theta):
    x, y = lib.generate_xy_loc(n, 3)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg(theta, x, y)
    S = np.tril(M.to_numpy())
    info = M.potrf()
    return M, S, info


@pytest.mark.parametrize("n,ts", [(1, 64), (63, 64), (65, 64), (128, 64), (129, 128), (191, 192), (193, 64),
                                  (321, 320), (449, 448), (705, 704), (961, 960), (1100, 1024), (1281, 128)])
def test_factor_small(lib, n, ts):
    """max |L L^T - S| <= 8 (n + 64) eps: the backward error of a Cholesky
    factorisation is (n + 1) eps sqrt(s_ii s_jj) (s_ii = 1), and the products
    with 64 x 64 inverses add 64 eps times the condition of such a block of L
    (below 8 for this covariance)."""
    M, S, info = _factor(lib, n, ts, (1.0, 0.1, 0.5))
    assert info == 0
    L = M.to_numpy()
    M.close()
    assert np.all(np.triu(L, 1) == 0.0)
    R = np.tril(L @ L.T - S)
    assert np.max(np.abs(R)) <= 8 * (n + 64) * EPS


@pytest.mark.parametrize("n,ts", [(12800, 320), (12801, 960), (13500, 1024)])
def test_factor_around_the_switch(lib, n, ts):
    """One launch for all 200 blocks, then a first tile step before it: L L^T v
    against S v for a vector of signs, whose rounding adds up over n terms."""
    M, S, info = _factor(lib, n, ts, (1.0, 0.1, 0.5))
    assert info == 0
    L = M.to_numpy()
    M.close()
    v = np.where(np.random.default_rng(0).random(n) < 0.5, -1.0, 1.0)
    Sv = S @ v + S.T @ v - np.diag(S) * v
    LLv = L @ (L.T @ v)
    # |error| <= 8 (n + 64) eps per entry of S, signs at random: sqrt(n) of
    # them, and five standard deviations
    assert np.max(np.abs(LLv - Sv)) <= 5 * np.sqrt(n) * 8 * (n + 64) * EPS


@pytest.mark.parametrize("n,ts,bad", [(300, 64, 0), (300, 64, 17), (300, 64, 64), (300, 64, 299), (1000, 320, 700)])
def test_first_failing_column(lib, n, ts, bad):
    """The first pivot that is not positive is the one reported."""
    x, y = lib.generate_xy_loc(n, 3)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg((1.0, 0.1, 0.5), x, y)
    S = M.to_numpy()
    S[bad, bad] = -1.0
    M.from_numpy(S)
    assert M.potrf() == bad + 1
    # the counters are back at zero: the next factorisation is a good one
    M.dcmg((1.0, 0.1, 0.5), x, y)
    assert M.potrf() == 0
    M.close()


@pytest.mark.parametrize("n,ts", [(700, 128), (1300, 320), (2000, 192)])
def test_mixed_panels(lib, n, ts):
    """Panels with FP32 and FP64 tiles (row groups end at tile boundaries):
    every tile forced to FP64 gives the FP64 likelihood, FP32 off-diagonal
    tiles one within their storage rounding, 2^-24 per entry of Sigma over an
    inverse whose trace is below 100 n."""
    from oracle import likelihood
    x, y = lib.generate_xy_loc(n, 4)
    z = np.sin(40.0 * x) * np.cos(31.0 * y)
    theta = (1.0, 0.05, 0.5)
    ref, ld, dp = likelihood.dmle("univariate_matern_stationary", x, y, z, np.array(theta))
    m = lib.ExactMLE(x, y, ts, precision=2)
    m.set_z(z)
    m.set_mixed(fp64_corr=1e-300)
    val = m.loglik(theta)
    assert abs(val - ref) <= 1e-11 * (abs(ld) + abs(dp))
    m.set_mixed()
    m.loglik(theta)
    assert abs(m.logdet - ld) <= 100 * n * 2.0 ** -24
    m.close()


@pytest.mark.parametrize("n,ts", [(2, 64), (65, 64), (129, 128), (257, 64), (641, 640), (1025, 192)])
def test_right_hand_side_row(lib, n, ts):
    """The forward solve inside the factorisation: quadratic form and
    log-determinant against the oracle, at sizes where the right-hand sides'
    row is the only one below a block column and where row groups are not
    full; 1e-11 of the larger of the two sums, as for the condition numbers
    up to 1e4 here; a second evaluation gives the same bits."""
    from oracle import likelihood
    x, y = lib.generate_xy_loc(n, 4)
    z = np.sin(40.0 * x) * np.cos(31.0 * y)
    theta = (1.0, 0.05, 0.8)
    ref, ld, dp = likelihood.dmle("univariate_matern_stationary", x, y, z, np.array(theta))
    m = lib.ExactMLE(x, y, ts)
    m.set_z(z)
    val = m.loglik(theta)
    first = (val, m.logdet, m.dotp)
    scale = max(abs(ld), abs(dp))
    assert abs(m.logdet - ld) <= 1e-11 * scale and abs(m.dotp - dp) <= 1e-11 * scale
    assert (m.loglik(theta), m.logdet, m.dotp) == first
    m.close()
