"""The BF16 update classes at every block shape (192, 128 and 64 rows) and at
the shortest and ordinary sums (one slice pair, and K = ts up to 960)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KN = "univariate_matern_nuggets_stationary"


@pytest.fixture(scope="module")
def lib():
    import exageostat_amd
    assert exageostat_amd.device_count() >= 1, "no HIP device visible"
    return exageostat_amd


@pytest.mark.parametrize("n,ts", [(400, 64), (900, 128), (1000, 192), (1500, 256), (1700, 320), (2000, 384), (2900, 960)])
@pytest.mark.parametrize("split", [1, 3, 4])
def test_logdet(lib, n, ts, split):
    """S = R + I (row norms of L: sqrt 2).  Operands rounded to a relative u
    change an entry of an off-diagonal tile by at most 2 u sum_k |L_ik| |L_jk|
    <= 4 u, and the log-determinant by sum |S^-1_ij| |dS_ij| over those tiles, to
    first order (factor 2 for the rest).  u = 2^-9 for single BF16 operands;
    split ones keep 2^-17, the dropped lo lo product and the FP32 sums and
    storage another 2^-16."""
    x, y = lib.generate_xy_loc(n, 11)
    th = (1.0, 0.05, 0.5, 1.0)
    M = lib.DeviceMatrix(n, n, ts, lower=True)
    M.dcmg(th[:3], x, y)
    S = np.tril(M.to_numpy())
    M.close()
    S = S + np.tril(S, -1).T + np.eye(n)
    off = np.abs(np.linalg.inv(S))
    for k in range(0, n, ts):
        off[k:k + ts, k:k + ts] = 0.0
    u = 2.0 ** -9 if split == 1 else 2.0 ** -15
    m = lib.ExactMLE(x, y, ts, kernel=KN, precision=2)
    m.set_z(np.sin(40.0 * x))
    m.set_mixed(fp32_corr=2.0 if split == 1 else 0.0, bf16=split == 1, lolo=split == 4)
    m.loglik(th)
    got = m.logdet
    m.close()
    assert abs(got - np.linalg.slogdet(S)[1]) <= 2 * 4 * u * off.sum()
