"""GPU: a small grid set up and rotated while little of the device's memory is
free is grouped, and as fast as elsewhere: what its tiles need is compared with
what is free, not with a share of the device."""

import ctypes as C
import time

import numpy as np
import pytest

from subsweep_amd import Sweep
from subsweep_amd import _native as N
from subsweep_amd import workloads as W
from subsweep_amd.sweep import rotation_matrix

pytestmark = pytest.mark.gpu


def test_small_grid_on_a_nearly_full_device(hip_available):
    N.sweep_lib()
    hip = C.CDLL("libamdhip64.so.7")  # the library's own runtime

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    pb = W.jittered_problem(12, 1.0, "4", 16, levels=2, periodic=True, steps=2, precision=32)
    turn = rotation_matrix((0.0, 0.0, 1.0), 0.3)

    def run():
        t0 = time.perf_counter()
        with Sweep(pb.params, pb.grid, *pb.state(), transport_mode=N.TRANSPORT_MODE_COMPILED) as s:
            t1 = time.perf_counter()
            fallback = [s.info().group_fallback]
            s.run_sweeps()
            t2 = time.perf_counter()
            s.rotate_directions(turn)
            t3 = time.perf_counter()
            fallback.append(s.info().group_fallback)
            s.run_sweeps()
            return fallback, t1 - t0 + t3 - t2, s.transport_state()

    roomy, _, want = run()
    hold = C.c_void_p()
    assert hip.hipMalloc(C.byref(hold), C.c_size_t(free_bytes() - (2 << 30))) == 0
    try:
        assert free_bytes() < (3 << 30)
        scarce, seconds, got = run()
    finally:
        assert hip.hipFree(hold) == 0
    assert roomy == scarce == [0, 0]
    assert seconds < 1.0  # a few milliseconds; a wait for memory takes two seconds each time
    for u, v in zip(got, want):
        assert np.array_equal(u.view(np.uint8), v.view(np.uint8))
