"""The staged pair sums with four lanes per target, and with one, against the
list-order kernel pinned through the autotuner: bit for bit, at the targets
per brick where the lanes change, with several shares of a brick, operand
counts that split into launches of 8, 4, 2 and 1, and operands whose records
exceed the LDS (smaller launches)."""
import math

import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def context(n, box, ne, periodic, prec, crowd=0):
    cfg = W._cfg([0, 0, 0], [box] * 3, periodic, [ne] * 3, precision=prec)
    rng = np.random.default_rng([n, crowd])
    x = rng.random((n, 3)) * box
    if crowd:  # some of them in one corner: bricks of several shares
        x[:crowd] *= 12.0 / box
    ctx = G.Context(cfg)
    ctx.reinit(x, rng.normal(size=(n, 3)))
    return ctx


def pin_lists(ctx, n, prec):
    lg = int(math.floor(math.log2(n)))
    p = "fp32c" if prec == G.FP32C else "fp64"
    for nr in (1, 2, 4, 8):
        ctx.tune_set("apply/%s/%d/%d" % (p, nr, lg), 0)
    for epi in (0, 1):
        ctx.tune_set("pair_beads/%s/%d/%d" % (p, epi, lg), 0)
    ctx.set_autotune(True)


@pytest.mark.parametrize("n,box,ne,periodic,crowd,nrhs,prec", [
    (5, 40.0, 20, (1, 1, 1), 0, 3, G.FP32C), (300, 40.0, 20, (1, 1, 0), 0, 16, G.FP32C),
    (2000, 64.0, 32, (1, 1, 1), 330, 15, G.FP32C), (2500, 64.0, 32, (0, 0, 0), 300, 1, G.FP32C),
    (9000, 64.0, 32, (1, 1, 1), 0, 8, G.FP32C), (10200, 64.0, 32, (1, 0, 1), 0, 2, G.FP32C),
    (4100, 48.0, 24, (1, 1, 1), 0, 7, G.FP32C), (3000, 100.0, 25, (1, 1, 1), 700, 4, G.FP32C),
    (300, 40.0, 20, (1, 1, 0), 0, 1, G.FP64), (2000, 64.0, 32, (1, 1, 1), 330, 1, G.FP64),
    (20000, 128.0, 64, (1, 1, 1), 0, 1, G.FP64), (21500, 128.0, 64, (1, 1, 1), 0, 1, G.FP64),
    (30000, 156.25, 40, (1, 1, 1), 400, 1, G.FP64)])  # bricks of about 240 targets, one over 512
def test_staged_sums_equal_the_list_order_kernel(n, box, ne, periodic, crowd, nrhs, prec):
    dw = G.normal(nrhs * 3 * n, 31).reshape(nrhs, n, 3)
    got = []
    for lists in (False, True):
        with context(n, box, ne, periodic, prec, crowd) as ctx:
            if lists:
                pin_lists(ctx, n, prec)
            u = ctx.combine_velocity()
            y, d, _ = ctx.cheb_brownian(5, 0.02, 3.0, dw, mode=G.CHEB_FIXED)
            ctx.set_graph(True)
            yg, dg, _ = ctx.cheb_brownian(5, 0.02, 3.0, dw, mode=G.CHEB_FIXED)
            got.append((u, y, d, yg, dg))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert np.array_equal(got[0][1], got[0][3]) and np.array_equal(got[0][2], got[0][4])


@pytest.mark.parametrize("n,crowd,prec", [(40, 0, G.FP64), (2500, 300, G.FP32C), (2500, 300, G.FP64),
                                          (12000, 0, G.FP32C)])
def test_reference_mode_staged_and_listed(n, crowd, prec):
    """The per-term estimators and the stop over different numbers of blocks:
    the same terms; the vectors differ only where the dot products' rounding
    could, that is not at all before the stop."""
    dw = G.normal(2 * 3 * n, 33).reshape(2, n, 3)
    got = []
    for lists in (False, True):
        with context(n, 64.0, 32, (1, 1, 0), prec, crowd) as ctx:
            if lists:
                pin_lists(ctx, n, prec)
            for _ in range(2):  # the second call starts from the first one's guess
                y, d, info = ctx.cheb_brownian(25, 0.004, 3.0, dw, tol=0.1, mode=G.CHEB_REFERENCE)
            got.append((y, d, [(i.terms, i.applies, i.converged) for i in info]))
    assert got[0][2] == got[1][2]
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
