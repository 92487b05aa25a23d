"""GPU: the grouped replay's cones where their tiles have edges, bitwise equal
to the geometric replay, which shares none of their layout: tasks with 4 to 115
upwind faces, cones with fewer tiles than a workgroup has waves and with more,
1 to 65 cells, restricted sweeps."""

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from test_gpu_direction_schedule import CASES, MYR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,roots", [(4, 64), (8, 32), (8, 128), (2, 32)])
@pytest.mark.parametrize("name,precision", [("tiny1", 64), ("tiny64", 32), ("tiny65", 64), ("hub13", 32), ("hub14", 64),
                                            ("hub115", 64), ("hub115", 32), ("slab110", 32)])
def test_cones_bitwise_equal_geometric(name, precision, levels, roots, hip_available):
    grid, dirs = CASES[name]()
    n = grid.num_cells
    rng = np.random.default_rng(2)
    src = np.where(rng.random(n) < 0.2, 10.0 ** rng.uniform(48, 50, n), 0.0)
    src[: min(n, 120)] = 1e49
    state = (1e-27 * np.exp(rng.standard_normal(n)), np.full(n, 1e-10), np.full(n, 1e4), src)
    p = SweepParameters(directions=dirs, num_timestep_levels=3, max_timestep=1e-3 * MYR,
                        transport_precision=precision)
    with Sweep(p, grid, *state, transport_mode=N.TRANSPORT_MODE_GEOMETRIC) as a, \
         Sweep(p, grid, *state, transport_mode=N.TRANSPORT_MODE_COMPILED, group_levels=levels,
               group_block=roots) as b:
        info = b.info()
        if info.group_fallback:
            assert info.group_tasks == 0 and name.startswith("slab")
        else:
            assert info.group_levels == levels and info.group_tasks >= n * len(dirs)
        for step in range(3):
            assert a.run_sweeps() == b.run_sweeps()
            for u, v in zip(a.transport_state(), b.transport_state()):
                assert np.array_equal(u.view(np.uint8), v.view(np.uint8)), f"step {step}"
            assert np.array_equal(a.results().level, b.results().level)


def test_cones_of_few_directions_stay_grouped(hip_available):
    """262144 cells x 16 directions: level sets of 3700 tasks on average, whose
    cones of 8 level sets do not all fit; the groups are then built with 8 only
    where level sets are narrow. Its memory stays within the estimate."""
    from subsweep_amd import workloads as W
    from subsweep_amd.serve import estimate_device_bytes
    pb = W.jittered_problem(64, 1.0, "6", 16, periodic=True, steps=2, precision=32)
    with Sweep(pb.params, pb.grid, *pb.state(), transport_mode=N.TRANSPORT_MODE_GEOMETRIC) as a, \
         Sweep(pb.params, pb.grid, *pb.state(), transport_mode=N.TRANSPORT_MODE_COMPILED) as b:
        info = b.info()
        assert info.group_fallback == 0 and info.group_tasks >= pb.grid.num_cells * 16
        for step in range(2):
            assert a.run_sweeps() == b.run_sweeps()
            for u, v in zip(a.transport_state(), b.transport_state()):
                assert np.array_equal(u.view(np.uint8), v.view(np.uint8)), f"step {step}"
        b.results()
    with Sweep(pb.params, pb.grid, *pb.state(), transport_mode=N.TRANSPORT_MODE_COMPILED) as b:
        b.run_sweeps()
        b.results()
        assert b.info().peak_device_bytes <= estimate_device_bytes(pb, N.TRANSPORT_MODE_COMPILED)
