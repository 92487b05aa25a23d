"""GPU: the chemistry's queue beyond its first round. k_chemistry_tail starts
2048 waves of 16 quads: up to 8192 queued cells get four quads each, up to 16384
two, more get one, and beyond 32768 the quads take further cells; as the queue
runs out, the quads of a row join into larger teams. The queued cells (those
whose full step the host's solver rejects) are counted here and asserted to lie
where each of those forms runs.

Bar as in test_gpu_chemistry_tail.py: 1e-10 relative for the state, process
counts within a handful of cells."""

import ctypes as C
import pathlib
import shutil
import subprocess

import numpy as np
import pytest

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import grid as G
from subsweep_amd import workloads as W

from parity_util import limiting_counts, summed_rate

MYR = 3.15576e13
HEADER = pathlib.Path(__file__).parent.parent / "subsweep_amd" / "csrc" / "chemistry.h"
SOURCE = f"""
#include "{HEADER}"
extern "C" int64_t solve(int64_t n, double* x, double* T, const double* rho, const double* vol, const double* len,
                         const double* rate, double dt, double safety, double* ts, int32_t* proc, int32_t* failed) {{
    int64_t rejected = 0;
    for (int64_t c = 0; c < n; c++) {{
        ssw::Cell cell;
        cell.x = x[c]; cell.T = T[c]; cell.rho = rho[c]; cell.vol = vol[c]; cell.len = len[c]; cell.rate = rate[c];
        cell.a = 1.0;
        const ssw::Floor floor{{true, cell.T, cell.x}};
        ssw::Walk w;
        w.dt = dt;
        bool ended = ssw::walk_step(cell, floor, dt, safety, w, ssw::Serial());
        rejected += !ended;
        while (!ended) ended = ssw::walk_step(cell, floor, dt, safety, w, ssw::Serial());
        x[c] = cell.x; T[c] = cell.T; ts[c] = w.ts; proc[c] = w.proc; failed[c] = w.failed;
    }}
    return rejected;
}}
"""


@pytest.fixture(scope="module")
def solver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("solver")
    (d / "solver.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", str(d / "solver.cpp"), "-o",
                    str(d / "solver.so")], check=True)
    lib = C.CDLL(str(d / "solver.so"))
    lib.solve.restype = C.c_int64

    def solve(x, T, rho, vol, size, rate, dt, safety):
        x, T = x.copy(), T.copy()
        n = x.size
        ts, proc, failed = np.empty(n), np.empty(n, np.int32), np.empty(n, np.int32)
        p = [np.ascontiguousarray(a, np.float64) for a in (rho, vol, size, rate)]
        ptr = lambda a: a.ctypes.data_as(C.c_void_p)
        rejected = lib.solve(C.c_int64(n), ptr(x), ptr(T), *(ptr(a) for a in p), C.c_double(dt), C.c_double(safety),
                             ptr(ts), ptr(proc), ptr(failed))
        return x, T, ts, proc, failed, rejected

    return solve


def problem(n):
    grid = G.cartesian_grid(n, W.BOX * n / 64, False)
    cells = grid.num_cells
    rng = np.random.default_rng(n)
    rho = W.RHO_MEAN * 10.0 ** rng.uniform(-3, 1, cells)
    x = 10.0 ** rng.uniform(-9, -0.01, cells)
    T = 10.0 ** rng.uniform(2, 5, cells)
    return grid, rho, x, T, 10.0 ** rng.uniform(44, 50, cells)


@pytest.mark.gpu
@pytest.mark.parametrize("n,low,high", [(29, 8192, 16384), (40, 16384, 32768), (48, 32768, 2 ** 31)])
@pytest.mark.parametrize("precision", [32, 64])
def test_long_queues_equal_the_hosts_solver(n, low, high, precision, solver, hip_available):
    grid, rho, x, T, src = problem(n)
    p = SweepParameters(directions=1, max_timestep=1e-2 * MYR, transport_precision=precision)
    with Sweep(p, grid, rho, x, T, src) as s:
        s.run_sweeps()
        r, info = s.results(), s.info()
        rate = summed_rate(s, src, 1)
    hx, hT, ts, proc, failed, rejected = solver(x, T, rho, grid.volume, grid.size, rate, p.max_timestep,
                                                p.chemistry_timestep_safety_factor)
    assert low < rejected <= high, "the queue's length"
    assert not failed.any() and int(info.chemistry_failures) == 0
    assert np.max(np.abs(r.ionized_hydrogen_fraction - hx) / hx) < 1e-10
    assert np.max(np.abs(r.temperature - hT) / hT) < 1e-10
    # the rate was 0 before: its timescale is dt (a change by the whole rate)
    assert (rate > 0).all()
    change = np.minimum(p.max_timestep, ts)
    counted = change < p.max_timestep
    got = limiting_counts(info)
    for k, name in enumerate(("temperature", "ionization_fraction")):
        assert abs(got[name] - int((counted & (proc == k)).sum())) <= 2 + rate.size // 10000
