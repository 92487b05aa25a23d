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
