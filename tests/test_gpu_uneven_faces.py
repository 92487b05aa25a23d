"""GPU: grids on which one side of a local face repeats it. Every face has its
mirror, so they are accepted, and the neighbour's upwind counter is decremented
once more than it counts; no other cell's counter may feel that, whichever
neighbours share a word with it.

Expected: along +x the level sets are those of the grid without the repeated
faces (each cell's only upwind neighbour is the same), and all launch shapes
give the geometric replay's bits. Along a diagonal, cells may become ready before
one of their upwind neighbours: the photon rate is then still the sum over the
present upwind rates, as the flux hook pulls it."""

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from subsweep_amd import grid as G
from subsweep_amd import workloads as W

pytestmark = pytest.mark.gpu

MYR = 3.15576e13


def repeated(n, cells, times):
    """The cartesian grid of n^3 cells, the +x face of `cells` repeated."""
    g = G.cartesian_grid(n, W.BOX * n / 64, False)
    plus_x = g.offsets[cells] + 1
    take = np.arange(g.num_faces)
    take = np.sort(np.concatenate([take, np.repeat(plus_x, times)]))
    off = g.offsets.copy()
    for c in cells:
        off[c + 1:] += times
    return g, G.Grid(off, g.neighbour[take], g.kind[take], g.area[take], g.normal[take], g.volume, g.size)


@pytest.mark.parametrize("times", [1, 5])
@pytest.mark.parametrize("shape", [{}, {"group_levels": 8}, {"group_levels": 1}, {"direction_sweeps": True}])
def test_repeated_faces_leave_other_cells_alone(shape, times, hip_available):
    n = 6
    cells = np.array([c for c in range(n ** 3) if c < (n - 1) * n * n and c % 3 == 0])  # not the last x plane
    plain, grid = repeated(n, cells, times)
    cells = plain.num_cells
    rng = np.random.default_rng(4)
    state = (W.RHO_MEAN * 10.0 ** rng.uniform(-3, 0, cells), np.full(cells, 1e-10), np.full(cells, 1e4),
             np.where(rng.random(cells) < 0.2, 1e48, 0.0))
    p = SweepParameters(directions=[[1.0, 0.0, 0.0]] * 3, num_timestep_levels=2, max_timestep=1e-3 * MYR)
    with Sweep(p, plain, *state) as a, Sweep(p, grid, *state, transport_mode=N.TRANSPORT_MODE_GEOMETRIC) as b, \
         Sweep(p, grid, *state, transport_mode=N.TRANSPORT_MODE_COMPILED, **shape) as s:
        for lvl in range(2):
            assert np.array_equal(s.levelsets(lvl), a.levelsets(lvl))
        assert s.levelsets(0).max() == n - 1
        for _ in range(2):
            assert b.run_sweeps() == s.run_sweeps()
            for u, v in zip(b.transport_state(), s.transport_state()):
                assert np.array_equal(u.view(np.uint8), v.view(np.uint8))
            assert np.array_equal(b.results().photon_rate, s.results().photon_rate)


@pytest.mark.parametrize("mode", [N.TRANSPORT_MODE_GEOMETRIC, N.TRANSPORT_MODE_COMPILED])
def test_photon_rate_is_pulled(mode, hip_available):
    n = 6
    cells = np.array([c for c in range(n ** 3) if c < (n - 1) * n * n and c % 3 == 0])
    _, grid = repeated(n, cells, 1)
    count = grid.num_cells
    state = (np.full(count, W.RHO_MEAN * 1e-3), np.full(count, 1e-10), np.full(count, 1e4), np.full(count, 1e48))
    h = np.sqrt(0.5)
    p = SweepParameters(directions=[[1.0, 0.0, 0.0], [h, h, 0.0]], max_timestep=1e-3 * MYR)
    with Sweep(p, grid, *state, transport_mode=mode) as s:
        for _ in range(2):
            s.run_sweeps()
            inc = s.fluxes()[0]
            assert np.array_equal(s.results().photon_rate, inc[0] + inc[1])
