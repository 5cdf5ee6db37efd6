"""The neighbour build's ways to the lists: one wave per target or one lane
per target (by a brick's targets and the stencil's rows), several blocks per
brick, the counters a build leaves clear for the next, empty and tiny
stores.  Local velocities against the oracle (FP64 to 1e-12, FP32C to 1e-6
relative L2: the suite's bars) and pair counts exactly."""
import numpy as np
import pytest

import copss_ggem as G
import oracle as O
import workloads as W
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def config(box, ne, periodic=(1, 1, 1)):
    return W._cfg([0, 0, 0], [box] * 3, periodic, [ne] * 3)


def oracle_mesh(cfg):
    return O.Mesh({k: cfg[k] for k in ("mu", "alpha", "box_min", "box_max", "periodic", "n_elem")}
                  | {"keep_stale_lists": 0})


def compare(ctx, cfg, x, f):
    ctx.reinit(x, f)
    m = oracle_mesh(cfg)
    m.reinit(x, f)
    off, _ = m.csr()
    assert ctx.neighbor_pairs() == int(off[-1])
    u = m.local_velocity_beads()
    for prec, bar in ((G.FP64, 1e-12), (G.FP32C, 1e-6)):
        ctx.set_precision(prec)
        got = ctx.local_velocity_beads()
        if np.linalg.norm(u) > 0:
            assert rel_l2(got, u) <= bar, prec
        else:
            assert not got.any()
    ctx.set_precision(G.FP64)


# beads, box, elements per axis: the bricks' targets lie below and above four
# per stencil row (69 rows at two-unit elements, 21 at four), in one or
# several shares of 32, with remainders of the 8-cell bricks
@pytest.mark.parametrize("n,box,ne,periodic", [
    (1, 40.0, 20, (1, 1, 1)), (2, 40.0, 20, (0, 0, 0)), (65, 38.0, 19, (1, 0, 1)), (2100, 46.0, 23, (1, 1, 1)),
    (2300, 48.0, 24, (1, 1, 0)), (3900, 100.0, 25, (1, 1, 1)), (1300, 64.0, 16, (0, 1, 1)),
    (700, 97.0, 25, (1, 1, 1))])
def test_lists_by_wave_and_by_lane(n, box, ne, periodic):
    cfg = config(box, ne, periodic)
    rng = np.random.default_rng(n)
    x = rng.random((n, 3)) * box
    with G.Context(cfg) as ctx:
        compare(ctx, cfg, x, rng.normal(size=(n, 3)))


def test_crowded_brick_beside_sparse_ones():
    """One brick above the rule and its neighbours below it."""
    cfg = config(64.0, 32)
    rng = np.random.default_rng(5)
    x = np.concatenate([rng.random((330, 3)) * 16.0, rng.random((400, 3)) * 64.0])
    with G.Context(cfg) as ctx:
        compare(ctx, cfg, x, rng.normal(size=x.shape))


def test_builds_in_turn_start_clear():
    """A build after a failed one, after a CSR export and after other sizes
    gives what a new context gives."""
    cfg = config(48.0, 24)
    rng = np.random.default_rng(9)
    sets = [rng.random((n, 3)) * 48.0 for n in (500, 37, 900)]
    f = [rng.normal(size=x.shape) for x in sets]
    with G.Context(cfg) as ctx:
        ctx.reinit(sets[0], f[0])
        ctx.neighbor_csr()
        bad = sets[0].copy()
        bad[3, 1] = 60.0
        with pytest.raises(G.GGEMError):
            ctx.reinit(bad, f[0])
        for x, fx in zip(sets + sets[:1], f + f[:1]):
            compare(ctx, cfg, x, fx)
        ctx.reinit(np.zeros((0, 3)), np.zeros((0, 3)))
        assert ctx.neighbor_pairs() == 0
        compare(ctx, cfg, sets[1], f[1])
