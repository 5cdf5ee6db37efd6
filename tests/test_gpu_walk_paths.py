"""Field points by sixteen lanes (lists in LDS, and the walk beyond their 128
entries), the outside flag they share with the build, and the element lists
by rows of eight elements, by elements in crowded boxes and at ragged grid
edges, against the oracle (FP64 to 1e-12, FP32C to 1e-6 relative L2: the
suite's bars)."""
import numpy as np
import pytest

import copss_ggem as G
import oracle as O
import workloads as W
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def setup(n, box, ne, periodic, crowd):
    cfg = W._cfg([0, 0, 0], [box] * 3, periodic, [ne] * 3)
    rng = np.random.default_rng([n, ne, crowd])
    x = rng.random((n, 3)) * box
    x[:crowd] = 0.3 * box + rng.random((crowd, 3)) * 4.0
    f = rng.normal(size=(n, 3))
    m = O.Mesh({k: cfg[k] for k in ("mu", "alpha", "box_min", "box_max", "periodic", "n_elem")}
               | {"keep_stale_lists": 0})
    m.reinit(x, f)
    ctx = G.Context(cfg)
    ctx.reinit(x, f)
    return cfg, x, f, m, ctx, rng


@pytest.mark.parametrize("n,box,ne,periodic,crowd,m", [
    (1, 40.0, 20, (1, 1, 1), 0, 17), (300, 40.0, 20, (1, 1, 0), 0, 1), (400, 41.0, 19, (0, 1, 1), 127, 300),
    (600, 40.0, 13, (1, 1, 1), 200, 257), (3000, 40.0, 20, (1, 1, 1), 0, 333)])
def test_points(n, box, ne, periodic, crowd, m):
    cfg, x, f, mesh, ctx, rng = setup(n, box, ne, periodic, crowd)
    with ctx:
        pts = rng.random((m, 3)) * box
        pts[: m // 3] = np.clip(x[rng.integers(0, n, m // 3)] + rng.normal(size=(m // 3, 3)), 0.0, box)
        pts[-1] = x[0]  # on a particle
        el = np.minimum((pts / (box / ne)).astype(np.int64), ne - 1)
        want = mesh.local_velocity_points(pts, (el[:, 0] + ne * (el[:, 1] + ne * el[:, 2])).astype(np.int32))
        for prec, bar in ((G.FP64, 1e-12), (G.FP32C, 1e-6)):
            ctx.set_precision(prec)
            assert rel_l2(ctx.local_velocity_points(pts), want) <= bar
        ctx.neighbor_csr()  # leaves the build's counters set
        bad = np.concatenate([pts, [[box + 1.0, 1.0, 1.0]]])
        with pytest.raises(G.GGEMError):
            ctx.local_velocity_points(bad)
        assert rel_l2(ctx.local_velocity_points(pts), want) <= 1e-6
        with pytest.raises(G.GGEMError):
            ctx.local_velocity_points(bad)
        ctx.reinit(x, f)  # the flag of the points is not the build's
        assert rel_l2(ctx.local_velocity_points(pts), want) <= 1e-6


@pytest.mark.parametrize("n,box,ne,periodic,crowd", [
    (1, 40.0, 20, (1, 1, 1), 0), (500, 40.0, 20, (1, 1, 0), 0), (700, 42.0, 17, (0, 0, 0), 60),
    (2500, 40.0, 20, (1, 1, 1), 2200), (400, 48.0, 12, (1, 0, 1), 100)])
def test_element_lists(n, box, ne, periodic, crowd):
    cfg, x, f, mesh, ctx, rng = setup(n, box, ne, periodic, crowd)
    with ctx:
        IF = G.hex20_if_table(ctx.consts().h, 2)
        rho_o, Fe_o = mesh.spread(2, IF)
        for prec, bar in ((G.FP64, 1e-12), (G.FP32C, 1e-6)):
            ctx.set_precision(prec)
            rho, Fe = ctx.spread(2, IF)
            assert rel_l2(rho, rho_o) <= bar and rel_l2(Fe, Fe_o) <= bar
