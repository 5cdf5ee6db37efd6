"""The staged FP64 pair sums of one operand against the list-order kernel
pinned through the autotuner, bit for bit, where the split changes: quads below
22,000 beads, blocks of 256 lanes above, of 512 in dense bricks or few.  Some
bricks hold more targets than a block has threads, or more records than the LDS.
And the list-order kernel, the default in sparse bricks, against the staged one."""
import math

import numpy as np
import pytest

import copss_ggem as G
from test_gpu_quad_paths import context, pin_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,box,ne,periodic,crowd", [
    (21999, 144.0, 72, (1, 1, 1), 0), (22000, 144.0, 72, (1, 1, 1), 900), (22001, 144.0, 72, (0, 1, 0), 600),
    (23000, 200.0, 65, (1, 1, 0), 300), (150000, 281.0, 72, (1, 1, 1), 700), (24000, 130.0, 64, (1, 1, 1), 900),
    (22500, 144.0, 72, (1, 1, 1), 6000)])
def test_fp64_blocks_equal_the_list_order_kernel(n, box, ne, periodic, crowd):
    dw = G.normal(3 * n, 37).reshape(1, n, 3)
    got = []
    for lists in (False, True):
        with context(n, box, ne, periodic, G.FP64, crowd) as ctx:
            if lists:
                pin_lists(ctx, n, G.FP64)
            u = ctx.combine_velocity()
            y, d, _ = ctx.cheb_brownian(5, 0.02, 3.0, dw, mode=G.CHEB_FIXED)
            ctx.set_graph(True)
            yg, dg, _ = ctx.cheb_brownian(5, 0.02, 3.0, dw, mode=G.CHEB_FIXED)
            got.append((u, y, d, yg, dg))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert np.array_equal(got[0][1], got[0][3]) and np.array_equal(got[0][2], got[0][4])


@pytest.mark.parametrize("n,box,ne,periodic", [(20000, 256.0, 128, (1, 1, 1)), (60000, 310.0, 100, (0, 1, 0))])
def test_fp64_sparse_bricks_default_equals_the_staged_kernel(n, box, ne, periodic):
    dw = G.normal(3 * n, 41).reshape(1, n, 3)
    lg = int(math.floor(math.log2(n)))
    got = []
    for staged in (False, True):
        with context(n, box, ne, periodic, G.FP64) as ctx:
            if staged:
                ctx.tune_set("apply/fp64/1/%d" % lg, 5)
                for epi in (0, 1):
                    ctx.tune_set("pair_beads/fp64/%d/%d" % (epi, lg), 5)
                ctx.set_autotune(True)
            u = ctx.combine_velocity()
            y, d, _ = ctx.cheb_brownian(5, 0.02, 3.0, dw, mode=G.CHEB_FIXED)
            yr, dr, info = ctx.cheb_brownian(12, 0.02, 3.0, dw, tol=1e-30, mode=G.CHEB_REFERENCE)
            got.append((u, y, d, yr, dr))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
