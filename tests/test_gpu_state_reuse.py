"""GPU: a state uploaded to a grid that has already been stepped, with another
state, gives the bits of a fresh handle: nothing of the former one is left in
the buffers, in any launch shape, with a negative source before it and after a
checkpoint was loaded."""

import numpy as np
import pytest

from subsweep_amd import Sweep
from subsweep_amd import _native as N
from subsweep_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [{}, {"direction_sweeps": True}, {"group_levels": 1},
                                   {"transport_mode": N.TRANSPORT_MODE_GEOMETRIC}])
@pytest.mark.parametrize("precision", [32, 64])
def test_new_state_equals_a_fresh_handle(shape, precision, hip_available):
    pb = W.jittered_problem(8, 1.0, "4", 16, levels=2, periodic=True, steps=3, precision=precision)
    pb = pb.with_params(max_timestep=1e-3 * 3.15576e13)
    rho, x, T, src = pb.state()
    other = src.copy()
    other[100] = -1e45  # small: a negative rate takes the solver millions of sub-steps
    with Sweep(pb.params, pb.grid, rho * 1e-3, x, T * 2, other, **shape) as a, \
         Sweep(pb.params, pb.grid, rho, x, T, src, **shape) as b:
        for first in (True, False):
            for _ in range(3):
                a.run_sweeps()
            a.results()
            if not first:
                a.load_checkpoint(a.save_checkpoint())
            a.upload_state(rho, x, T, src)
            if not first:
                b.upload_state(rho, x, T, src)
            for step in range(3):
                assert a.run_sweeps() == b.run_sweeps()
                for u, v in zip(a.transport_state(), b.transport_state()):
                    assert np.array_equal(u.view(np.uint8), v.view(np.uint8)), f"step {step}"
                ra, rb = a.results(), b.results()
                for f in ("ionized_hydrogen_fraction", "temperature", "timestep", "photon_rate", "level",
                          "change_timescale"):
                    assert np.array_equal(getattr(ra, f), getattr(rb, f)), f
                assert a.info().updates_last_step == b.info().updates_last_step
