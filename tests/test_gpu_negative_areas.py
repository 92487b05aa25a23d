"""GPU: the photon rate on a grid with negative face areas, where an incoming
rate can be negative although no source is: it is the pull over the present
upwind rates that the flux hook gives, not the rates that were clamped when
they were stored."""

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from subsweep_amd import grid as G
from subsweep_amd import workloads as W

pytestmark = pytest.mark.gpu

MYR = 3.15576e13


@pytest.mark.parametrize("shape", [{}, {"direction_sweeps": True}, {"transport_mode": N.TRANSPORT_MODE_GEOMETRIC}])
@pytest.mark.parametrize("precision", [32, 64])
def test_photon_rate_with_negative_areas(shape, precision, hip_available):
    n = 5
    grid = G.cartesian_grid(n, W.BOX * n / 64, False)
    c = (1 * n + 2) * n + 2             # its +x face, and the mirror face, with a negative area
    nb = c + n * n
    assert grid.neighbour[6 * c + 1] == nb and grid.neighbour[6 * nb] == c
    grid.area[[6 * c + 1, 6 * nb]] *= -0.1
    cells = grid.num_cells
    src = np.zeros(cells)
    src[c] = 1e49
    h = np.sqrt(0.5)
    p = SweepParameters(directions=[[h, h, 0.0], [h, 0.0, h]], max_timestep=1e-3 * MYR, transport_precision=precision)
    with Sweep(p, grid, np.full(cells, W.RHO_MEAN * 1e-4), np.full(cells, 1e-10), np.full(cells, 1e4), src,
               **shape) as s:
        for _ in range(2):
            s.run_sweeps()
            inc = s.fluxes()[0]
            assert (inc[:, nb] < 0.0).any()
            for noalloc in (False, True):
                assert np.array_equal(s.results(noalloc=noalloc).photon_rate, inc[0] + inc[1])


@pytest.mark.parametrize("shape", [{}, {"direction_sweeps": True}, {"transport_mode": N.TRANSPORT_MODE_GEOMETRIC}])
@pytest.mark.parametrize("precision", [32, 64])
def test_photon_rate_after_a_checkpoint_with_negative_rates(shape, precision, hip_available):
    # a checkpoint whose sources are zeroed after a negative one has left
    # negative rates behind: the sources say nothing of what the first sweeps read
    grid = G.voronoi_grid(G.uniform_points(300, W.BOX, 11), W.BOX)
    cells, dirs = grid.num_cells, 16
    src = np.full(cells, 1e47)
    src[cells // 2] = -1e48
    p = SweepParameters(directions=dirs, num_timestep_levels=3, periodic=False, max_timestep=1e-3 * MYR,
                        significant_rate_threshold=-1e60,  # else a negative rate is not passed on
                        transport_precision=precision)
    state = (np.full(cells, W.RHO_MEAN * 1e-4), np.full(cells, 1e-10), np.full(cells, 1e4))
    with Sweep(p, grid, *state, src, **shape) as a, Sweep(p, grid, *state, np.full(cells, 1e47), **shape) as b:
        a.run_sweeps()
        assert (a.fluxes()[0] < 0.0).any()
        buf = bytearray(a.save_checkpoint())
        real = precision // 8
        header = len(buf) - (64 * cells + (cells + 7) // 8 * 8 + 2 * dirs * cells * real)
        at = header + 3 * 8 * cells
        buf[at:at + 8 * cells] = np.full(cells, 1e46 / dirs).tobytes()
        b.load_checkpoint(bytes(buf))
        for _ in range(4):
            inc = b.fluxes()[0]
            want = np.zeros(cells)
            for d in range(dirs):
                want = want + inc[d]
            for noalloc in (False, True):
                assert np.array_equal(b.results(noalloc=noalloc).photon_rate, want)
            b.run_sweeps()
