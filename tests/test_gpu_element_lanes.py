"""Element lists a lane per element, where stencil rows are few (five-unit
elements: 13, six-unit: 9) or hold many beads: ragged grid edges, periodic
wraps of rows, lists past a block's LDS buffer.  rho and Fe against the
oracle (FP64 to 1e-12, FP32C to 1e-6 relative L2: the suite's bars)."""
import numpy as np
import pytest

import copss_ggem as G
import oracle as O
import workloads as W
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,ne,periodic,crowd", [
    (1, 60.0, 12, (1, 1, 1), 0), (300, 55.0, 11, (1, 1, 0), 0), (2000, 95.0, 19, (0, 1, 1), 500),
    (1500, 78.0, 13, (1, 0, 1), 400), (900, 45.0, 9, (0, 0, 0), 0),
    (67000, 218.4, 56, (1, 1, 1), 0)])  # 195 beads a brick, 21 rows
def test_lists_by_element(n, box, ne, periodic, crowd):
    cfg = W._cfg([0, 0, 0], [box] * 3, periodic, [ne] * 3)
    rng = np.random.default_rng([n, ne])
    x = rng.random((n, 3)) * box
    x[:crowd] = box * 0.96 + rng.random((crowd, 3)) * box * 0.039  # in the last elements
    f = rng.normal(size=(n, 3))
    m = O.Mesh({k: cfg[k] for k in ("mu", "alpha", "box_min", "box_max", "periodic", "n_elem")}
               | {"keep_stale_lists": 0})
    m.reinit(x, f)
    with G.Context(cfg) as ctx:
        ctx.reinit(x, f)
        IF = G.hex20_if_table(ctx.consts().h, 2)
        rho_o, Fe_o = m.spread(2, IF)
        for prec, bar in ((G.FP64, 1e-12), (G.FP32C, 1e-6)):
            ctx.set_precision(prec)
            rho, Fe = ctx.spread(2, IF)
            assert rel_l2(rho, rho_o) <= bar and rel_l2(Fe, Fe_o) <= bar
