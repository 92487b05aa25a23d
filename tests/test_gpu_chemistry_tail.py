"""GPU: the chemistry's two kernels against the host's solver (the same code,
cell after cell): cells that take one step and cells that take many sub-steps,
at cell counts around a quad's wave (16 cells) and beyond the queue's first
round (2048 waves), so that quads take further cells.

Bar: 1e-10 relative, as everywhere for the FP64 chemistry (the device's and the
host's exp and pow differ by an ulp or so, which the sub-steps carry on; the
number of sub-steps agrees unless a relative change lies within that of the
safety factor). Process counts within the same handful of cells."""

import ctypes as C

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from subsweep_amd import grid as G
from subsweep_amd import workloads as W

from parity_util import limiting_counts, summed_rate

pytestmark = pytest.mark.gpu

MYR = 3.15576e13


@pytest.mark.parametrize("n,quiet", [(1, False), (2, True), (3, False), (11, False), (34, False)])
@pytest.mark.parametrize("precision", [32, 64])
def test_chemistry_equals_the_hosts_solver(n, quiet, precision, hip_available):
    grid = G.cartesian_grid(n, W.BOX * n / 64, False)
    cells = grid.num_cells
    rng = np.random.default_rng(n)
    rho = W.RHO_MEAN * 10.0 ** rng.uniform(-3, 1, cells)
    x = 10.0 ** rng.uniform(-9, -0.01, cells)
    T = 10.0 ** rng.uniform(2, 5, cells)
    src = np.zeros(cells) if quiet else 10.0 ** rng.uniform(44, 50, cells)
    p = SweepParameters(directions=1, max_timestep=1e-2 * MYR, transport_precision=precision)
    lib = N.sweep_lib()
    with Sweep(p, grid, rho, x, T, src) as s:
        s.run_sweeps()
        r, info = s.results(), s.info()
        rate = summed_rate(s, src, 1)
    counts = dict.fromkeys(("temperature", "ionization_fraction", "photon_rate"), 0)
    worst = 0.0
    for c in range(cells):
        st = np.array([x[c], T[c]])
        proc, failed = C.c_int32(), C.c_int32()
        ts = lib.ssw_chemistry_timestep(N.ptr(st, C.c_double), rho[c], grid.volume[c], grid.size[c], rate[c], 1.0, 1,
                                        p.max_timestep, p.chemistry_timestep_safety_factor, C.byref(proc),
                                        C.byref(failed))
        assert failed.value == 0
        got = (r.ionized_hydrogen_fraction[c], r.temperature[c])
        worst = max(worst, abs(got[0] - st[0]) / st[0], abs(got[1] - st[1]) / st[1])
        # the rate was 0 before: its timescale is dt (a change by the whole rate) unless there is none
        rate_ts = p.max_timestep if rate[c] > 0 else p.max_timestep * 2.0 ** -52
        change = rate_ts if rate_ts < ts else ts
        if change < p.max_timestep:
            counts[("temperature", "ionization_fraction")[proc.value] if rate_ts >= ts else "photon_rate"] += 1
    assert worst < 1e-10
    assert int(info.chemistry_failures) == 0
    got = limiting_counts(info)
    for k, v in counts.items():
        assert abs(got[k] - v) <= 2 + cells // 10000, (got, counts)
