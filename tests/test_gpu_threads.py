"""First evaluations of several threads at once, each with its own context: the
launch parameters that they share are worked out once."""
from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THETA = (1.0, 0.1, 0.5)


def test_four_contexts_at_once():
    import exageostat_amd as lib
    x, y = lib.generate_xy_loc(300, 5)
    z = np.sin(40.0 * x)
    models = [lib.ExactMLE(x, y, 64) for _ in range(4)]
    for m in models:
        m.set_z(z)
    out = [None] * len(models)
    start = threading.Barrier(len(models))

    def work(i):
        start.wait()
        out[i] = models[i].loglik(THETA, grad=True)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(models))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for m in models:
        m.close()
    for ll, g in out[1:]:
        assert ll == out[0][0] and np.array_equal(g, out[0][1])
