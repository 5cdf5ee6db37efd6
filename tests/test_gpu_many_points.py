"""Field points past the most threads of one launch (2^28 points of sixteen
lanes): a block of points repeated gives its results repeated, bit for bit.
6.4 GB of points and of results."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def test_points_past_one_launch():
    cfg, x, f = W.make_inputs("beads100")
    with G.Context(cfg) as ctx:
        ctx.reinit(x, f)
        k = 1 << 20
        block = np.random.default_rng(5).random((k, 3)) * 40.0
        want = ctx.local_velocity_points(block)
        m = (1 << 28) + 5
        pts = np.empty((m, 3))
        for i in range(0, m, k):
            pts[i:i + k] = block[:m - i]
        got = ctx.local_velocity_points(pts)
        del pts
        for i in range(0, m, k):
            assert np.array_equal(got[i:i + k], want[:m - i]), i
