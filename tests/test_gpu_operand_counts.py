"""Several noise vectors at once, in every launch size they split into (8, 4,
2, 1) and both layouts of the gather records: each vector's step is what it
is alone, bit for bit.  With the staged kernels, with bricks that are not
staged, under the explicit minimum image, through graph replay, and with the
kept vectors applied again after a rebuild."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu

N, BOX = 1100, 48.0


def context(prec, state):
    rng = np.random.default_rng(17)
    x = rng.random((N, 3)) * BOX
    if state == "crowded":
        x[:500] = 4.0 + rng.random((500, 3)) * 6.0
    if state == "unstaged":  # a box over the staged records, and lists of hundreds
        x[:] = 20.0 + rng.random((N, 3)) * 8.0
        x = np.concatenate([x, x[:, ::-1] + 0.125])
    f = rng.normal(size=x.shape)
    ctx = G.Context(W._cfg([0, 0, 0], [BOX] * 3, [1, 1, 0], [24, 24, 24], precision=prec))
    ctx.reinit(x, f)
    if state == "moved":
        ctx.update_positions(np.where(np.arange(3) == 0, (x + 0.7) % BOX, x), f)
    return ctx, x, f


@pytest.mark.parametrize("prec", [G.FP64, G.FP32C])
@pytest.mark.parametrize("state", ["plain", "crowded", "unstaged", "moved"])
@pytest.mark.parametrize("nrhs", [2, 3, 4, 7, 8, 13, 16])
def test_vectors_together_equal_vectors_alone(prec, state, nrhs):
    ctx, x, f = context(prec, state)
    with ctx:
        dw = G.normal(nrhs * x.size, 23).reshape(nrhs, -1, 3)
        step = lambda w: ctx.cheb_brownian(5, 0.02, 30.0, w, mode=G.CHEB_FIXED, keep=True)[:2]
        alone = [step(w[None]) for w in dw]
        y, d = step(dw)
        for r in range(nrhs):
            assert np.array_equal(y[r], alone[r][0][0]) and np.array_equal(d[r], alone[r][1][0]), r
        assert np.array_equal(ctx.displacement_apply(), d)
        ctx.set_graph(True)
        for _ in range(3):
            yg, dg = step(dw)
            assert np.array_equal(yg, y) and np.array_equal(dg, d)
        ctx.set_graph(False)
        if state != "moved":  # the kept vectors at other positions, against each alone there
            x2 = np.where(np.arange(3) == 1, (x + 0.9) % BOX, x)
            ctx.reinit(x2, f)
            d2 = ctx.displacement_apply()
            for r in (0, nrhs - 1):
                ctx.set_forces(y[r])
                assert np.array_equal(d2[r], ctx.mobility_apply(None)), r


# 70,000 beads: 70, 137 and 137 beads a brick, the last with remainders of the
# 8-cell bricks and walls; two, four and eight vectors a lane per target
@pytest.mark.parametrize("box,ne,periodic,nrhs", [
    (240.0, 80, (1, 1, 1), 3), (249.6, 64, (1, 1, 1), 4), (249.6, 64, (1, 1, 1), 16), (241.8, 62, (1, 0, 1), 11)])
def test_dense_bricks_equal_the_list_order_kernel(box, ne, periodic, nrhs):
    n = 70000
    rng = np.random.default_rng(ne)
    x, f = rng.random((n, 3)) * box, rng.normal(size=(n, 3))
    dw = G.normal(nrhs * 3 * n, 29).reshape(nrhs, n, 3)
    got = []
    for lists in (False, True):
        with G.Context(W._cfg([0, 0, 0], [box] * 3, periodic, [ne] * 3, precision=G.FP32C)) as ctx:
            ctx.reinit(x, f)
            if lists:
                for nr in (1, 2, 4, 8):
                    ctx.tune_set("apply/fp32c/%d/16" % nr, 0)
                ctx.set_autotune(True)
            got.append(ctx.cheb_brownian(3, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2])
            ctx.set_graph(True)
            got.append(ctx.cheb_brownian(3, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2])
    for y, d in got[1:]:
        assert np.array_equal(y, got[0][0]) and np.array_equal(d, got[0][1])


@pytest.mark.parametrize("nrhs", [2, 4, 8, 13])
def test_sparse_and_dense_builds_in_turn(nrhs):
    """Several FP32C vectors on one context through builds that change their
    route: 8,000 beads over 6,200 bricks (list order), the same beads in a
    corner (staged), over the bricks again; the captured step follows.  Each
    step against the staged kernels pinned, and against one vector alone."""
    n, ne, h = 8000, 200, 2.0
    rng = np.random.default_rng(nrhs)
    wide = rng.random((n, 3)) * ne * h
    sets = [wide, wide * 0.2, wide]
    f = rng.normal(size=(n, 3))
    dw = G.normal(nrhs * 3 * n, 37).reshape(nrhs, n, 3)
    step = lambda c, w: c.cheb_brownian(4, 0.02, 3.0, w, mode=G.CHEB_FIXED)[:2]
    cfg = W._cfg([0, 0, 0], [ne * h] * 3, [1, 1, 1], [ne] * 3, precision=G.FP32C)
    with G.Context(cfg) as ctx, G.Context(cfg) as staged:
        for nr in (1, 2, 4, 8):
            staged.tune_set("apply/fp32c/%d/12" % nr, 5)
        staged.set_autotune(True)
        for x in sets:
            ctx.reinit(x, f)
            staged.reinit(x, f)
            want = step(staged, dw)
            ctx.set_graph(False)
            got = step(ctx, dw)
            ctx.set_graph(True)
            for y, d in (got, step(ctx, dw), step(ctx, dw)):
                assert np.array_equal(y, want[0]) and np.array_equal(d, want[1])
            one = step(ctx, dw[:1])
            assert np.array_equal(one[0][0], want[0][0]) and np.array_equal(one[1][0], want[1][0])


@pytest.mark.parametrize("n,ne,h", [(101000, 80, 3.9), (101000, 96, 3.1)])
def test_one_vector_many_beads(n, ne, h):
    """One FP32C vector on either side of the rule at 100,000 beads (101 and 59
    a brick) against the list-order kernel."""
    rng = np.random.default_rng(ne)
    x, f = rng.random((n, 3)) * ne * h, rng.normal(size=(n, 3))
    dw = G.normal(3 * n, 41).reshape(1, n, 3)
    got = []
    for lists in (False, True):
        with G.Context(W._cfg([0, 0, 0], [ne * h] * 3, [1, 1, 0], [ne] * 3, precision=G.FP32C)) as ctx:
            ctx.reinit(x, f)
            if lists:
                for key in ("apply/fp32c/1/16", "pair_beads/fp32c/0/16"):
                    ctx.tune_set(key, 0)
                ctx.set_autotune(True)
            got.append((ctx.local_velocity_beads(), *ctx.cheb_brownian(3, 0.02, 3.0, dw, mode=G.CHEB_FIXED)[:2]))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
