"""Record and list fills of many beads, where a brick's targets per stencil row
choose a wave or a lane per target: bricks on either side of the limit in one
system, with 69, 29 and 21 rows.  Pair counts exactly, local velocities against
the oracle (FP64 to 1e-12, FP32C to 1e-6), the list-order kernel bit for bit."""
import numpy as np
import pytest

import copss_ggem as G
from test_gpu_build_paths import compare, config
from test_gpu_quad_paths import pin_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ne,h,power,periodic", [
    (24000, 40, 2.0, 1.0, (1, 1, 1)), (40000, 56, 2.0, 1.5, (1, 1, 0)), (40000, 57, 3.1, 1.3, (1, 1, 1)),
    (40000, 63, 3.9, 1.4, (0, 1, 1)), (17000, 48, 3.1, 1.0, (1, 1, 1))])
def test_fills_on_both_sides_of_the_limit(n, ne, h, power, periodic):
    cfg = config(ne * h, ne, periodic)
    rng = np.random.default_rng([n, ne])
    x, f = rng.random((n, 3)) ** power * ne * h, rng.normal(size=(n, 3))
    with G.Context(cfg) as ctx:
        compare(ctx, cfg, x, f)
        ctx.set_precision(G.FP32C)
        u = ctx.local_velocity_beads()
    with G.Context(cfg) as ctx:
        ctx.set_precision(G.FP32C)
        pin_lists(ctx, n, G.FP32C)
        ctx.reinit(x, f)
        assert np.array_equal(ctx.local_velocity_beads(), u)
