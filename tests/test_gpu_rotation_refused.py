"""GPU: a rotation whose directions have a dependency cycle is refused, and
the handle goes on as if it had not been asked: bitwise the steps of a handle
that was never rotated, in every launch shape, and the next rotation works."""

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from subsweep_amd.grid import Grid
from subsweep_amd.sweep import rotation_matrix

pytestmark = pytest.mark.gpu

SHAPES = {
    "default": {},
    "per level": {"group_levels": 1},
    "direction": {"direction_sweeps": True},
    "geometric": {"transport_mode": N.TRANSPORT_MODE_GEOMETRIC},
}


def triangle():
    """Three cells whose forward faces 0 -> 1 -> 2 -> 0 all look along +x: a
    cycle for the direction +x, none for +y."""
    s = np.sqrt(0.5)
    forward = {(0, 1): (1.0, 0.0, 0.0), (1, 2): (s, s, 0.0), (2, 0): (s, -s, 0.0)}
    faces = [[], [], []]
    for (a, b), n in forward.items():
        faces[a].append((b, n))
        faces[b].append((a, tuple(-v for v in n)))
    flat = [f for cell in faces for f in cell]
    return Grid(np.array([0, 2, 4, 6], np.int64), np.array([b for b, _ in flat], np.int32), np.zeros(6, np.uint8),
                np.full(6, 1e40), np.array([n for _, n in flat]), np.full(3, 1e60), np.full(3, 1e20))


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("precision", [32, 64])
def test_refused_rotation_leaves_the_handle(shape, precision, hip_available):
    state = (np.full(3, 1e-25), np.full(3, 1e-10), np.full(3, 1e4), np.array([1e49, 0.0, 0.0]))
    p = SweepParameters(directions=[[0.0, 1.0, 0.0], [0.0, 1.0, 0.0]], num_timestep_levels=2, max_timestep=1e10,
                        transport_precision=precision)
    quarter = rotation_matrix((0.0, 0.0, 1.0), -0.5 * np.pi)  # +y to +x
    half = rotation_matrix((0.0, 0.0, 1.0), np.pi)            # +y to -y
    with Sweep(p, triangle(), *state, **SHAPES[shape]) as a, Sweep(p, triangle(), *state, **SHAPES[shape]) as b:
        for step in range(4):
            with pytest.raises(N.SweepError) as e:
                b.rotate_directions(quarter)
            assert e.value.code == -4
            assert np.array_equal(a.levelsets(0), b.levelsets(0))
            assert a.info().downwind_local == b.info().downwind_local
            assert a.run_sweeps() == b.run_sweeps()
            for u, v in zip(a.transport_state(), b.transport_state()):
                assert np.array_equal(u.view(np.uint8), v.view(np.uint8)), f"step {step}"
            ra, rb = a.results(), b.results()
            assert np.array_equal(ra.photon_rate, rb.photon_rate) and np.array_equal(ra.temperature, rb.temperature)
        a.rotate_directions(half)
        b.rotate_directions(half)
        for _ in range(2):
            assert a.run_sweeps() == b.run_sweeps()
            for u, v in zip(a.fluxes(), b.fluxes()):
                assert np.array_equal(u, v)
