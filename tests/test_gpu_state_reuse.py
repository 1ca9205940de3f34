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
