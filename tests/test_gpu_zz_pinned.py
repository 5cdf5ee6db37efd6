"""ggem_local_velocity_points_noalloc allocates nothing, pinned host memory
included: a large call on a fresh context maps no further memory through the
device files."""
import ctypes as C

import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def device_mappings():
    """Bytes of this process mapped through the GPU's device files (pinned
    host memory and device memory alike)."""
    total = 0
    with open("/proc/self/maps") as fh:
        for line in fh:
            span, _, rest = line.partition(" ")
            if "/dev/dri/" in rest or "/dev/kfd" in rest:
                lo, hi = span.split("-")
                total += int(hi, 16) - int(lo, 16)
    return total


def test_noalloc_allocates_no_pinned_memory():
    cfg, x, f = W.make_inputs("beads100")
    fn = G.lib().ggem_local_velocity_points_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p]
    pts = np.random.default_rng(3).random((65536, 3)) * 40.0
    u = np.zeros_like(pts)
    with G.Context(cfg) as first, G.Context(cfg) as ctx:
        for c in (first, ctx):
            c.reinit(x, f)
        # the first context's call loads the kernels and fills the runtime's own staging
        assert fn(first._h, len(pts), pts.ctypes.data, None, u.ctypes.data) == 0
        before = device_mappings()
        assert before > 0
        assert fn(ctx._h, len(pts), pts.ctypes.data, None, u.ctypes.data) == 0
        assert device_mappings() == before
        assert np.array_equal(u, ctx.local_velocity_points(pts))
