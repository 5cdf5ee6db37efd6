"""Readbacks of a context whose device is not the calling thread's current
one: the pinned buffers' events belong to the context's device."""
import ctypes as C

import numpy as np
import pytest

import copss_ggem as G
import workloads as W

pytestmark = pytest.mark.gpu


def test_readback_with_another_current_device():
    hip = C.CDLL("libamdhip64.so")
    count = C.c_int()
    if hip.hipGetDeviceCount(C.byref(count)) != 0 or count.value < 2:
        pytest.skip("needs two devices")
    cfg, x, f = W.make_inputs("beads20k", n=40000)
    with G.Context(dict(cfg, device=0)) as ctx:
        ctx.set_particles(x, f)
        assert hip.hipSetDevice(1) == 0
        try:
            assert np.array_equal(ctx.get_positions()[0], x)  # 0.96 MB: several pieces
        finally:
            hip.hipSetDevice(0)
