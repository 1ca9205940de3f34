"""Kriging whose C22 is factored in one launch with the forward solve inside
(Context::factor_solve), whose right-hand side row is shared with the
likelihood's larger matrix of the same context."""
import numpy as np
import pytest

from oracle import datagen, likelihood

pytestmark = pytest.mark.gpu

K = "univariate_matern_stationary"
THETA = (1.0, 0.1, 0.5)


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    exageostat_amd.load()
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


@pytest.mark.parametrize("nobs", [1, 63, 64, 65, 321, 700])
def test_after_a_larger_evaluation(lib, nobs):
    """1,000 rows evaluated with a z of NaN first: nothing of it is left in
    the padding of the smaller matrix.  1e-9 of the largest prediction, the
    bound of the other kriging tests."""
    x, y, _ = datagen.generate_xy_loc(1024, 7)
    z = np.random.default_rng(7).standard_normal(1024)
    m = lib.ExactMLE(x[:1000], y[:1000], 320)
    m.set_z(np.full(1000, np.nan))
    m.loglik(THETA)
    miss = slice(1000, 1024)
    zm, _ = m.predict(THETA, x[:nobs], y[:nobs], z[:nobs], x[miss], y[miss], z[miss])
    m.close()
    ref = likelihood.predict(K, x[:nobs], y[:nobs], z[:nobs], x[miss], y[miss], THETA, z[miss])[0]
    assert np.max(np.abs(zm - ref)) <= 1e-9 * np.max(np.abs(ref))


def test_before_a_larger_evaluation(lib):
    """The buffers of 300 rows grow for 1,000: the likelihood as without the
    kriging before it."""
    x, y, _ = datagen.generate_xy_loc(1024, 8)
    x, y = x[:1000], y[:1000]
    z = np.random.default_rng(8).standard_normal(1000)
    m = lib.ExactMLE(x, y, 320)
    m.set_z(z)
    m.predict(THETA, x[:300], y[:300], z[:300], x[300:310], y[300:310], z[300:310])
    val = m.loglik(THETA)
    m.close()
    ref = likelihood.dmle(K, x, y, z, THETA)[0]
    assert abs(val - ref) <= 1e-9 * abs(ref)
