"""Builds whose scans take more than one pass: meshes over 4096 scan tiles
(8.4M cells) and over 65,536 bricks, stores over 65,536 slices, with and
without particles.  The beads of a region far smaller than the mesh have the
lists they have in a mesh of that region alone, so velocities and steps agree
bit for bit (positions are multiples of 2^-20: moving them by whole elements
is exact, and a list's order does not depend on where the bricks begin)."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def config(ne, h, prec):
    return W._cfg([0, 0, 0], [h * k for k in ne], [0, 0, 0], ne, precision=prec)


def region(n, edge, seed):
    rng = np.random.default_rng(seed)
    x = np.floor(rng.random((n, 3)) * edge * 2.0 ** 20) / 2.0 ** 20
    return x, rng.normal(size=(n, 3))


@pytest.mark.parametrize("prec", [G.FP64, G.FP32C])
@pytest.mark.parametrize("ne", [(208, 208, 208), (1024, 1024, 40)])
def test_mesh_over_the_scan_limits(ne, prec):
    x, f = region(1500, 40.0, 3)
    dw = G.normal(2 * x.size, 9).reshape(2, -1, 3)
    with G.Context(config((20, 20, 20), 2.0, prec)) as ctx:
        ctx.reinit(x, f)
        pairs, u = ctx.neighbor_pairs(), ctx.combine_velocity()
        d = ctx.cheb_brownian(6, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[1]
    with G.Context(config(ne, 2.0, prec)) as ctx:
        ctx.reinit(np.zeros((0, 3)), np.zeros((0, 3)))  # no particles yet
        assert ctx.neighbor_pairs() == 0
        # at the first corner, at the last one (far past the first pass of
        # every scan), without particles again, in the middle
        at = [(0, 0, 0), tuple(k - 20 for k in ne), None, tuple(8 * (k // 16) - 8 for k in ne)]
        for c in at:
            if c is None:
                ctx.reinit(np.zeros((0, 3)), np.zeros((0, 3)))
                assert ctx.neighbor_pairs() == 0
                continue
            ctx.reinit(x + 2.0 * np.array(c), f)
            assert ctx.neighbor_pairs() == pairs
            assert np.array_equal(ctx.combine_velocity(), u)
            assert np.array_equal(ctx.cheb_brownian(6, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[1], d)


def test_store_over_the_scan_limit():
    """4.25M beads (66,407 slices), four-unit elements."""
    n, ne, h = 4250000, 256, 4.0
    x, f = region(n, ne * h, 4)
    keep = np.all(x < 128.0, axis=1)
    inner = np.all(x[keep] < 128.0 - 16.0, axis=1)  # lists that end inside the region
    assert inner.sum() > 2000
    with G.Context(config((32, 32, 32), h, G.FP32C)) as ctx:
        ctx.reinit(x[keep], f[keep])
        u = ctx.local_velocity_beads()[inner]
    with G.Context(config((ne,) * 3, h, G.FP32C)) as ctx:
        ctx.reinit(x, f)
        assert np.array_equal(ctx.local_velocity_beads()[keep][inner], u)
        ctx.set_precision(G.FP64)
        v = ctx.local_velocity_beads()[keep][inner]
        assert np.linalg.norm(v - u) <= 1e-6 * np.linalg.norm(v)
