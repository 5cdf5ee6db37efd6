"""The convergence-checked Chebyshev step over the block counts where its
decision changes hands: the launch's last block (up to 128 blocks), one
deciding block, several (over 8,192).  Terms, estimators and vectors against
the host-driven rule (a host operator that applies the same context's
mobility), the stop before the last term and never."""
import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ne,h,prec", [
    (60, 20, 2.0, G.FP64), (1000, 40, 2.0, G.FP32C), (1100, 48, 2.0, G.FP64), (2600, 40, 2.0, G.FP64),
    (30000, 200, 2.0, G.FP64), (30000, 200, 2.0, G.FP32C), (70000, 48, 3.9, G.FP32C)])
@pytest.mark.parametrize("tol", [0.05, 1e-30])
def test_decision_against_the_host_rule(n, ne, h, prec, tol):
    rng = np.random.default_rng([n, ne])
    x, f = rng.random((n, 3)) * ne * h, rng.normal(size=(n, 3))
    dw = G.normal(2 * 3 * n, 43).reshape(2, n, 3)
    cfg = W._cfg([0, 0, 0], [ne * h] * 3, [1, 1, 1], [ne] * 3, precision=prec)
    with G.Context(cfg) as ctx, G.Context(cfg) as other:
        ctx.reinit(x, f)
        other.reinit(x, f)
        for _ in range(2):  # the second call starts from the first one's stop
            y, d, info = ctx.cheb_brownian(20, 0.05, 3.0, dw, tol=tol, mode=G.CHEB_REFERENCE)
        yh, dh, ih = ctx.cheb_brownian(20, 0.05, 3.0, dw, tol=tol, mode=G.CHEB_REFERENCE,
                                       op=lambda v: other.mobility_apply(v.reshape(-1, 3)))
    bar = 1e-12 if prec == G.FP64 else 1e-6
    for r in range(2):
        assert info[r].terms == ih[r].terms and info[r].converged == ih[r].converged
        assert abs(info[r].err2 - ih[r].err2) <= bar * ih[r].err2
        assert np.linalg.norm(y[r] - yh[r]) <= bar * np.linalg.norm(yh[r])
        assert np.linalg.norm(d[r] - dh[r]) <= bar * np.linalg.norm(dh[r])
    assert (info[0].terms < 20) == (tol == 0.05)
