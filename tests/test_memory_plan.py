"""CPU: the decisions of the schedule build and of the request loop on device
memory (subsweep_amd/csrc/memory_plan.h, compiled here with the host compiler)."""

import pytest

from memory_plan_util import DIRECTIONS, GEOMETRIC, GROUPED, PER_LEVEL, build_plan

MB = 1 << 20
GB = 1 << 30


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    return build_plan(tmp_path_factory)


@pytest.mark.parametrize("tiles,later,free,fits", [
    (4 * MB, 1 * MB, 7 * MB, True),             # a small grid on a nearly full device
    (4 * MB, 1 * MB, 5 * MB, False),
    (0, 0, 1 * MB, True),
    (200 * GB, 20 * GB, 222 * GB, True),        # the largest
    (200 * GB, 20 * GB, 221 * GB, False),
    (200 * GB, 0, 202 * GB, True),              # its state is there already (a rotation)
    (150 * GB, 0, 0, False),
])
def test_cones_fit(plan, tiles, later, free, fits):
    assert bool(plan.cones_fit(tiles, later, free)) == fits


@pytest.mark.parametrize("rs", [4, 8])
def test_later_allocations(plan, rs):
    n, d, per = 1000, 16, 100
    state = plan.state_bytes(n, n * d, per * d, rs)
    assert state == 2 * n * d * rs + per * d * rs + n * (80 + 2 * rs + 4)
    assert plan.offset_bytes(n * d, per * d, rs) == (n + per) * d * rs


# cells, faces, periodic cells, directions, levels, FP32: estimate of a compiled
# request while all held planes and the group lists of every timestep level
ADMITTED = [
    (1000, 6000, 0, 16, 1, False, 11041568),
    (4096, 63000, 1400, 1, 1, True, 10452023),
    (8192, 127000, 2000, 16, 1, True, 31806763),
    (32768, 508000, 6000, 84, 4, True, 491294785),
    (262144, 4040000, 24000, 84, 1, True, 3326914344),
    (262144, 4040000, 24000, 84, 4, False, 6291717486),
    (524288, 8080000, 40000, 32, 2, True, 2950719832),
    (2097152, 32300000, 100000, 84, 4, True, 30016745761),
]


@pytest.mark.parametrize("case", ADMITTED)
def test_a_compiled_launch_shape_fits_where_planes_and_lists_did(plan, case):
    *problem, before = case
    assert plan.handle_bytes(*problem, DIRECTIONS) <= before
    assert plan.handle_bytes(*problem, PER_LEVEL) <= before
    assert plan.handle_bytes(*problem, GEOMETRIC) <= plan.handle_bytes(*problem, PER_LEVEL)
    # cones that do not fit leave planes
    assert plan.handle_bytes(*problem, GROUPED) >= plan.handle_bytes(*problem, PER_LEVEL)
    assert plan.replay_bytes(*problem, GROUPED) < plan.handle_bytes(*problem, GROUPED)
