"""The phases of an evaluation whose factorisation, forward solve and sums are
one sequence of launches: each has a time, and together they are the whole."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ts", [(1, 64), (400, 64), (1600, 320)])
def test_phases_add_up(n, ts):
    import exageostat_amd as lib
    x, y = lib.generate_xy_loc(n, 5)
    m = lib.ExactMLE(x, y, ts)
    m.set_z(np.sin(40.0 * x))
    for _ in range(2):  # the second evaluation allocates nothing
        m.loglik((1.0, 0.1, 0.8))
    t = m.phase_times()
    m.close()
    parts = [t[k] for k in ("gen", "facto", "logdet", "solve")]
    assert all(p > 0.0 for p in parts), t
    assert abs(sum(parts) - t["total"]) <= 1e-12 * t["total"]
