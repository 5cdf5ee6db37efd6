"""Calls whose route depends on what the context went through before:
captured graphs and tuned launch shapes met again after the positions moved
on kept lists or after a fuller build.  Each result is compared with that of
a context without the graph or the tuner, bit for bit (the routes sum the
same terms in the same order)."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def context(n, box, ne, prec, seed=3):
    rng = np.random.default_rng([n, ne, seed])
    x = rng.random((n, 3)) * box
    f = rng.normal(size=(n, 3))
    ctx = G.Context(W._cfg([0, 0, 0], [box] * 3, [1, 1, 1], [ne] * 3, precision=prec))
    ctx.reinit(x, f)
    return ctx, x, f


def moved(x, box):
    """Every bead a third of a unit along x, wrapped into the box."""
    y = x + np.array([0.35, 0.0, 0.0])
    y[:, 0] -= box * (y[:, 0] >= box)
    return y


@pytest.mark.parametrize("prec", [G.FP32C, G.FP64])
@pytest.mark.parametrize("nrhs", [1, 2])
def test_graph_after_update_positions(prec, nrhs):
    """One-unit elements: no brick's box fits the staged kernels, before and
    after the move.  Beads that crossed a face keep lists with the shifts of
    the build, so the step after the move takes the explicit minimum image."""
    n, box = 400, 24.0
    dw = G.normal(nrhs * 3 * n, 5).reshape(nrhs, n, 3)
    got = []
    for graph in (False, True):
        ctx, x, f = context(n, box, 24, prec)
        with ctx:
            ctx.set_graph(graph)
            steps = []
            for _ in range(2):
                steps.append(ctx.cheb_brownian(8, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2])
            ctx.update_positions(moved(x, box), f)
            for _ in range(2):
                steps.append(ctx.cheb_brownian(8, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2])
            got.append(steps)
    for (ya, da), (yb, db) in zip(*got):
        assert np.array_equal(ya, yb) and np.array_equal(da, db)
    assert not np.array_equal(got[0][0][1], got[0][2][1])  # the move shows


def tuned_and_plain(n, box, ne, prec, then, nrhs=1, mode=None):
    """Steps and velocities of a context whose tuner has recorded the staged
    kernels, and of one without a tuner, after `then` changed both."""
    dw = G.normal(nrhs * 3 * n, 7).reshape(nrhs, n, 3)
    got = []
    for tune in (True, False):
        ctx, x, f = context(n, box, ne, prec)
        with ctx:
            if tune:
                ctx.set_autotune(True)
                lg = n.bit_length() - 1
                p = "fp32c" if prec == G.FP32C else "fp64"
                for key in ["apply/%s/%d/%d" % (p, nr, lg) for nr in ((1, 2, 4, 8) if prec == G.FP32C else (1,))] + \
                        ["pair_beads/%s/%d/%d" % (p, epi, lg) for epi in (0, 1)]:
                    ctx.tune_set(key, 5)  # what the tuner records where the staged kernels win
            run = lambda: (ctx.local_velocity_beads(), ctx.combine_velocity(),
                           *ctx.cheb_brownian(8, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2],
                           *ctx.cheb_brownian(8, 0.02, 3.0, dw, mode=G.CHEB_REFERENCE)[:2])
            run()
            then(ctx, x, f)
            got.append(run())
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec", [G.FP32C, G.FP64])
@pytest.mark.parametrize("nrhs", [1, 3, 8])
def test_tuned_shape_after_update_positions(prec, nrhs):
    """The explicit minimum image has no staged kernel."""
    tuned_and_plain(1500, 40.0, 20, prec, lambda ctx, x, f: ctx.update_positions(moved(x, 40.0), f), nrhs)


@pytest.mark.parametrize("prec", [G.FP32C, G.FP64])
@pytest.mark.parametrize("nrhs", [1, 2, 8])
def test_tuned_shape_after_a_fuller_build(prec, nrhs):
    """Beads gather in one corner: brick boxes with more records than the
    several operands' LDS holds, some with more than are staged at all."""
    def crowd(ctx, x, f):
        ctx.reinit(x * np.where(np.arange(len(x)) % 8 < 6, 0.3, 1.0)[:, None], f)

    tuned_and_plain(3000, 64.0, 32, prec, crowd, nrhs)


def test_nodes_past_the_mesh_are_zero():
    """Nodal results of a longer array than the mesh's nodes end in zeros."""
    ctx, x, f = context(200, 40.0, 20, G.FP64)
    with ctx:
        xyz, conn = G.hex20_box_mesh(ctx.cfg)
        n = len(xyz)
        ctx.set_fe_mesh(n, conn)
        IF = G.hex20_if_table(ctx.consts().h, 2)
        junk = np.full((n + 500, 3), 7.0)  # the allocation that the results may reuse
        want = ctx.spread_nodes(2, IF, n)
        del junk
        got = ctx.spread_nodes(2, IF, n + 500)
        assert np.array_equal(got[:n], want) and not got[n:].any()
        want = ctx.assemble_rhs(2, IF, G.rhs_opts(), n)
        junk = np.full((n + 500, 3), 7.0)
        del junk
        got = ctx.assemble_rhs(2, IF, G.rhs_opts(), n + 500)
        assert np.array_equal(got[:n], want) and not got[n:].any()
