"""Results copied to the host in pieces arrive whole: sizes around the smallest
piece's 512 KiB (21845.3 vectors of three doubles), around three of them and
eight (longer pieces from there on), odd remainders, several copies in turn."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2730, 21845, 21846, 65535, 65536, 65537, 87382, 150001, 174762, 174763, 800001])
def test_noise_round_trip(n):
    cfg = W._cfg([0, 0, 0], [400] * 3, [1, 1, 1], [100] * 3)
    with G.Context(cfg) as ctx:
        ctx.set_particles(np.full((n, 3), 1.0))
        for nrhs in (1, 2, 1):
            dw = G.normal(nrhs * 3 * n, 50 + nrhs).reshape(nrhs, n, 3)
            ctx.set_noise(dw)
            assert np.array_equal(ctx.get_noise(), dw)
