"""Rounding inside the dataflow factorisation: a long sum of small products is
not rounded at the magnitude of the entry that it is subtracted from."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ts", [(1100, 64), (5000, 320)])
def test_long_sums_of_small_products(n, ts):
    """Diagonal 101, sums of squares below it a few tenths: the residual
    101 - sum_k L_ik^2 of the last 512 rows (in extended precision) comes from
    the roundings at the diagonal's magnitude alone: one per 1,024 columns, four
    block products, 15 columns of a panel and the root twice, some 30 of
    ulp(101) / sqrt(12) rms each; twice that is allowed.  n roundings would be
    six times as much at n = 5,000."""
    import exageostat_amd as lib
    x, y = lib.generate_xy_loc(n, 3)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg((1.0, 0.03, 0.5, 100.0), x, y, kernel="univariate_matern_nuggets_stationary")
    assert M.potrf() == 0
    L = M.to_numpy()[-512:].astype(np.longdouble)
    M.close()
    res = 101.0 - np.sum(L * L, axis=1)
    rms = float(np.sqrt(np.mean(res * res)))
    assert rms <= 2 * np.sqrt(30) * np.spacing(101.0) / np.sqrt(12), rms
