"""Evaluations on a context that another kind of evaluation, or a failed one,
has used before: the results are those of a new context."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THETA = (1.0, 0.1, 0.5)


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


@pytest.mark.parametrize("n,ts", [(100, 64), (450, 64), (700, 320)])
def test_gradient_after_a_failed_band(lib, n, ts):
    """A band-limited evaluation that fails (a negative variance) leaves NaN in
    the padded rows of the solution; the exact gradient after it has the bits
    of one without it."""
    x, y = lib.generate_xy_loc(n, 5)
    z = np.sin(40.0 * x) * np.cos(31.0 * y)
    m = lib.ExactMLE(x, y, ts)
    m.set_z(z)
    ll, g = m.loglik(THETA, grad=True)
    assert np.isfinite(ll) and np.all(np.isfinite(g))
    m.data.computation = b"diag_approx"
    m.loglik((-1.0, 0.1, 0.5))
    assert m.status == 1
    m.data.computation = b"exact"
    ll2, g2 = m.loglik(THETA, grad=True)
    m.close()
    assert ll2 == ll and np.array_equal(g2, g)


@pytest.mark.parametrize("nobs,ts", [(100, 64), (700, 320)])
def test_kriging_after_a_failed_one(lib, nobs, ts):
    """A covariance that is not positive definite (a negative variance): the
    error is reported and the observations on the device are left alone; kriging
    and likelihood of the same context afterwards against the oracle, to 1e-9 of
    the largest prediction and of the likelihood, the bounds of their tests."""
    import ctypes

    from exageostat_amd import _lib
    from oracle import datagen, likelihood
    kernel = "univariate_matern_stationary"
    x, y, _ = datagen.generate_xy_loc(1024, 9)
    z = np.random.default_rng(9).standard_normal(1024)
    m = lib.ExactMLE(x[:1000], y[:1000], ts)
    m.set_z(z[:1000])
    miss = slice(1000, 1024)
    held = (x[:nobs], y[:nobs], z[:nobs], x[miss], y[miss], z[miss])
    with pytest.raises(RuntimeError, match="not positive definite"):
        m.predict((-1.0, 0.1, 0.5), *held)
    left = np.empty(nobs)
    desc = ctypes.cast(m.data.descZobs, ctypes.POINTER(_lib.Desc))
    m.lib.EXAGEOSTAT_Tile_to_Lapack(desc, left.ctypes.data_as(_lib.c_double_p), nobs)
    assert np.array_equal(left, z[:nobs])
    zm, _ = m.predict(THETA, *held)
    val = m.loglik(THETA)
    m.close()
    ref = likelihood.predict(kernel, x[:nobs], y[:nobs], z[:nobs], x[miss], y[miss], THETA, z[miss])[0]
    assert np.max(np.abs(zm - ref)) <= 1e-9 * np.max(np.abs(ref))
    ref = likelihood.dmle(kernel, x[:1000], y[:1000], z[:1000], THETA)[0]
    assert abs(val - ref) <= 1e-9 * abs(ref)
