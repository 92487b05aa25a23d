"""What the library is timed on: the calls that a radiative-transfer program makes through `subsweep_amd`.

Five kinds of pass, all through the public Python interface:

  frame   one `SweepPlugin.run_sweep_system` call of a running simulation: every sweep of the timestep
          levels, the chemistry, and the per-cell results back on the host. With `optional` the optional
          chemistry fields too; with `rotate` the directions turn after the call, as the parameter asks.
  solve   one request on a resident grid: the gas and its sources are uploaded, `steps` steps, the results
          (what the request loop does for a grid that it has already set up).
  packed  `problems` small independent simulations stepped together with `Sweep.run_sweeps_packed`, each one's
          results read back.
  cold    one request on a grid that the device has not seen: handle, grid upload and schedule, state, `steps`
          steps, results.

Grids: `cartesian` is the reference's cartesian test grid, `jittered` the Voronoi grid of a jittered lattice
(uniform resolution), `clustered` the Voronoi grid of points drawn from a lognormal field (cell volumes spanning
about 1e3). A grid depends on its sizes alone and is built once per process, as a program that solves many gas
states on it would keep it; density, sources and their luminosities come from the seed. `shape` is the launch
shape: the library's default, or direction sweeps, which the autotuner picks on the benchmark's workloads and
the serving benchmark asks for.
"""

from __future__ import annotations

import functools
import math

import numpy as np

from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import grid as G
from subsweep_amd import units as U
from subsweep_amd import workloads as W
from subsweep_amd.sweep import CHEMISTRY_OUTPUTS, SweepPlugin

DIRECTIONS = (16, 21, 32, 64, 84)  # the direction tables in use
WARM = 2  # frames already run when a simulation is timed: its timestep levels have settled


def listed():
    return [
        # The smallest call: the reference's cartesian test grid with open boundaries, where launches, host work
        # and the copies of the results are everything.
        case("frame", "cartesian", 1000, 16, name="frame_cartesian_1k_fp64", periodic=False),
        # The single-source problem of the tests and of the reference's example: 16 directions, FP64, with the
        # optional chemistry fields that its output lists.
        case("frame", "jittered", 32768, 16, name="frame_jittered_32k_fp64", sources=1, optional=True),
        # The benchmark's precision workload, in both transport precisions, launched as the autotuner chooses.
        case("frame", "jittered", 262144, 84, name="frame_jittered_262k_fp32", precision=32, shape="direction",
             threshold=1e-5),
        case("frame", "jittered", 262144, 84, name="frame_jittered_262k_fp64", shape="direction", threshold=1e-5),
        # The same kind of problem at an odd size for a user who tunes nothing.
        case("frame", "jittered", 117649, 64, name="frame_jittered_118k_fp32_default", precision=32),
        # The headline workload: 2 M clustered cells, 84 directions, four timestep levels, 1024 sources.
        case("frame", "clustered", 2097152, 84, name="frame_clustered_2m_fp32", levels=4, precision=32,
             shape="direction", sources=1024),
        # Requests of the serving mix on resident grids: a small and a middling one, with timestep levels.
        case("solve", "clustered", 23457, 32, name="solve_clustered_23k_fp32", levels=2, precision=32, steps=10,
             shape="direction", sources=17),
        case("solve", "jittered", 157464, 64, name="solve_jittered_157k_fp32", levels=4, precision=32, steps=10,
             shape="direction", sources=40),
        # Thin gas, where photons cross the box and the timestep levels spread over all four: sweeps restricted to
        # few active cells, FP64, default launch shape.
        case("solve", "clustered", 20000, 84, name="solve_thin_20k_fp64", levels=4, steps=5, sources=16, thin=True),
        # Eight small problems stepped together.
        case("packed", "jittered", 13824, 32, name="packed_8_fp32", precision=32, problems=8, sources=8),
        # A request on a grid seen for the first time: the schedule build is most of it.
        case("cold", "jittered", 32768, 84, name="cold_jittered_33k_fp32", precision=32, steps=2, shape="direction",
             sources=8),
        # A simulation with rotating directions: a new schedule every frame.
        case("frame", "jittered", 12167, 32, name="frame_rotating_12k_fp64", sources=4, rotate=True),
    ]


def case(kind, grid, cells, directions, name=None, levels=1, precision=64, periodic=True, shape="default", sources=64,
         threshold=0.0, steps=1, problems=1, thin=False, optional=False, rotate=False):
    c = {"kind": kind, "grid": grid, "cells": cells, "directions": directions, "levels": levels,
         "precision": precision, "periodic": periodic, "shape": shape, "sources": sources, "threshold": threshold,
         "steps": steps, "problems": problems, "thin": thin, "optional": optional, "rotate": rotate}
    return dict(c, name=name) if name else c


def draw(rng):
    """A case of the listed ranges: sizes over their logarithm up to the serving mix's largest grid."""
    kind = rng.choice(("frame", "frame", "frame", "solve", "solve", "solve", "packed", "cold"))
    grid = rng.choice(("cartesian", "jittered", "jittered", "clustered", "clustered"))
    rotate = kind == "frame" and rng.random() < 0.15
    most = {"frame": 524288, "solve": 262144, "packed": 27000, "cold": 65536}[kind]
    cells = int(math.exp(rng.uniform(math.log(900), math.log(20000 if rotate else most))))
    if grid != "clustered":
        cells = max(2, round(cells ** (1.0 / 3.0))) ** 3
    directions = rng.choice(DIRECTIONS)
    if directions * cells > 84 * 262144:
        directions = 21
    levels = rng.choice((1, 1, 2, 4)) if kind in ("solve", "cold") else 1
    precision = rng.choice((32, 32, 64))
    # rotations and packed steps are only offered with the default shape's options; the rest take either
    shape = "default" if rotate or kind == "packed" else rng.choice(("default", "direction", "direction"))
    return case(kind, grid, cells, directions, levels=levels, precision=precision,
                periodic=not (grid == "cartesian" and rng.random() < 0.5), shape=shape,
                sources=rng.randint(1, 64), threshold=rng.choice((0.0, 1e-5)),
                steps={"solve": rng.randint(3, 10), "cold": rng.randint(1, 3)}.get(kind, 1),
                problems=rng.randint(3, 8) if kind == "packed" else 1,
                thin=grid != "cartesian" and rng.random() < 0.3, optional=kind == "frame" and rng.random() < 0.2,
                rotate=rotate)


# ---------------------------------------------------------------------------------------------------------------
# inputs


@functools.lru_cache(maxsize=24)
def the_grid(kind, cells, periodic, field_seed=1340):
    """(grid, the density field at the cells or None); the clustered field's mesh follows the workloads'."""
    if kind == "clustered":
        pts, delta = G.clustered_points(cells, W.BOX, mesh=128 if cells > 524288 else 64, seed=field_seed)
        return G.voronoi_grid(pts, W.BOX), delta
    n = round(cells ** (1.0 / 3.0))
    if kind == "cartesian":
        return G.cartesian_grid(n, W.BOX, periodic), None
    return G.voronoi_grid(G.jittered_lattice(n, W.BOX, 0.3, field_seed - 2), W.BOX), None


def problem(c, seed, k=0):
    """The k-th problem of a case: (grid, parameters, density, ionised fraction, temperature, source)."""
    cells = c["cells"]
    if k and c["grid"] != "clustered":  # the problems of a pack differ in size
        cells = max(2, round(cells ** (1.0 / 3.0)) - 2 + k % 5) ** 3
    elif k:
        cells = cells - 97 * k if cells > 2000 else cells + 13 * k
    directions = c["directions"] if c["kind"] != "packed" else DIRECTIONS[(DIRECTIONS.index(c["directions"]) + k) % 5]
    g, delta = the_grid(c["grid"], cells, c["periodic"])
    n = g.num_cells
    rng = np.random.default_rng([seed, k])
    mean = W.RHO_MEAN * (1e-4 if c["thin"] else 1.0)
    noise = G.lognormal_density(n, 1.0, 1.0 if delta is None else 0.1, seed % (1 << 31) + k)
    rho = mean * noise * (1.0 if delta is None else delta)
    if c["grid"] == "clustered" and not c["thin"]:  # on the densest cells, p(L) ~ L^-2, escape fraction 0.01
        src = np.zeros(n)
        src[np.argsort(-rho, kind="stable")[:c["sources"]]] = 0.01 * W.power_law_luminosities(
            min(c["sources"], n), 1e48, 1e52, seed % (1 << 31) + k)
    else:  # at uniform positions, 10^U(48, 51) photons/s, on the nearest cells
        src, _ = G.assign_sources(g.points, rng.uniform(0.0, W.BOX, (c["sources"], 3)),
                                  10.0 ** rng.uniform(48.0, 51.0, c["sources"]))
    params = SweepParameters(directions=directions, num_timestep_levels=c["levels"], periodic=c["periodic"],
                             max_timestep=(1e-3 if c["thin"] else 1.0) * U.MEGAYEARS,
                             significant_rate_threshold=c["threshold"], timestep_safety_factor=0.1,
                             transport_precision=c["precision"])
    return g, params, rho, np.full(n, 1e-10), np.full(n, 1e4), src


def sweep(c, p):
    return Sweep(p[1], p[0], *p[2:], direction_sweeps=c["shape"] == "direction")


def prepare(case, seed):
    c = case
    if c["kind"] == "packed":
        s = [sweep(c, problem(c, seed, k)) for k in range(c["problems"])]
        for _ in range(WARM):
            Sweep.run_sweeps_packed(s)
        return {"case": c, "sweeps": s}
    p = problem(c, seed)
    if c["kind"] == "cold":
        return {"case": c, "problem": p}
    s = sweep(c, p)
    if c["kind"] == "solve":
        return {"case": c, "sweep": s, "gas": p[2:]}
    plugin = SweepPlugin(s, optional_outputs=CHEMISTRY_OUTPUTS if c["optional"] else (),
                         rotate_directions=c["rotate"])
    for _ in range(1 + WARM):  # the plugin's first call runs no sweeps
        plugin.run_sweep_system()
    return {"case": c, "plugin": plugin}


# ---------------------------------------------------------------------------------------------------------------
# one pass


def fields(r):
    return {"ionized_hydrogen_fraction": r.ionized_hydrogen_fraction, "temperature": r.temperature,
            "timestep": r.timestep, "photon_rate": r.photon_rate, "level": r.level,
            "change_timescale": r.change_timescale}


def run(state):
    c = state["case"]
    if c["kind"] == "frame":
        out = fields(state["plugin"].run_sweep_system())
        return dict(out, **state["plugin"].chemistry) if c["optional"] else out
    if c["kind"] == "packed":
        Sweep.run_sweeps_packed(state["sweeps"])
        return [fields(s.results()) for s in state["sweeps"]]
    if c["kind"] == "solve":
        s = state["sweep"]
        s.upload_state(*state["gas"])
    else:
        s = sweep(c, state["problem"])
    elapsed = [s.run_sweeps() for _ in range(c["steps"])]
    out = dict(fields(s.results()), time=float(sum(elapsed)))
    if c["kind"] == "cold":
        s.close()
    return out


def work(case):
    """The face lists once per sweep (a normal and an area in 64 bits and a neighbour), every cell's state in and
    out, and the rate of every cell and direction read and written once per sweep in the transport's precision;
    a multiplication and an addition per face for which side it is on, its weight and the sum. Sweeps below the
    deepest level are counted as full, which they nearly are where most cells sit on the deepest level."""
    c = case
    faces = 6.0 if c["grid"] == "cartesian" else 15.4
    sweeps = c["steps"] * 2 ** (c["levels"] - 1)
    n = c["cells"] * c["problems"]
    updates = n * c["directions"] * sweeps
    return {"bytes": int(n * sweeps * (faces * 36 + 16 * 8) + 2 * updates * c["precision"] // 8),
            "flops": int(updates * (faces * 7 + faces) + n * sweeps * 400)}


# ---------------------------------------------------------------------------------------------------------------
# the same in plain numpy, 64 bits: one timestep level, small grids


def exact(case, seed):
    c = case
    if (c["levels"] > 1 or c["rotate"] or c["kind"] == "packed" or c["cells"] * c["directions"] > 600000
            or c["cells"] * c["directions"] * (c["steps"] + WARM) > 3000000):
        return None
    g, prm, rho, x, T, src = problem(c, seed)
    dirs = direction_vectors(prm.directions)
    steps = WARM + 1 if c["kind"] == "frame" else c["steps"]
    n, D, dt = g.num_cells, len(dirs), prm.max_timestep
    off, kind = np.asarray(g.offsets), np.asarray(g.kind)
    owner = np.repeat(np.arange(n), np.diff(off))
    nb = np.asarray(g.neighbour).astype(np.int64)
    sod = src / D
    plans = [upwind_plan(g, owner, nb, kind, d) for d in dirs]
    X, P = [np.zeros(n) for _ in dirs], [np.zeros(n) for _ in dirs]
    for _ in range(steps):
        att = absorbed_not(rho, x, g.size)
        total, photons = np.zeros(n), np.zeros(n)
        for d, (order, starts, target, source, w, edge_starts, A, pt, ps, pw) in enumerate(plans):
            I = np.zeros(n)
            Xd = X[d]
            for k in range(len(starts) - 1):
                cells = order[starts[k]:starts[k + 1]]
                e = slice(edge_starts[k], edge_starts[k + 1])
                np.add.at(I, target[e], w[e] * Xd[source[e]])
                rate = (np.maximum(I[cells], 0.0) + sod[cells]) + P[d][cells]
                out = np.where(rate < prm.significant_rate_threshold, 0.0, rate * att[cells])
                Xd[cells] = np.where(A[cells] > 0.0, out / np.where(A[cells] > 0.0, A[cells], 1.0), 0.0)
            P[d] = np.bincount(pt, pw * Xd[ps], n) if len(pt) else P[d]
            photons += I
            total += (I + sod) + P[d]
        gas = Gas(rho, g.volume, g.size, total)
        x, T, used = gas.advance(x.copy(), T.copy(), dt, prm.chemistry_timestep_safety_factor)
    out = {"ionized_hydrogen_fraction": x, "temperature": T, "timestep": used, "photon_rate": photons, "level": None,
           "change_timescale": None}  # the change of a rate from one step to the next cancels: not a value to hold to
    if c["kind"] != "frame":
        out["time"] = float(steps * dt)
    if c["optional"]:
        year = 3.15576e7
        new = gas.newly_ionized(x, year)
        out["photoionization_rate"] = new / (gas.nh * (1.0 - x) * gas.vol) / year
        heat = new / gas.vol * (gas.PHOTON - gas.RYDBERG) / year
        out["heating_rate"] = heat - gas.cooling(x, T)
        out["recombination_rate"] = gas.alpha(T) * (gas.nh * x) * x
        out["collisional_ionization_rate"] = gas.beta(T) * (gas.nh * x) * (1.0 - x)
    return out


def direction_vectors(directions):
    from subsweep_amd.sweep import direction_table
    return direction_table(directions)  # data: the tabulated bins


def upwind_plan(g, owner, nb, kind, d):
    """Cells in an order in which each follows its upwind neighbours, level by level, with the edges into them."""
    dot = g.normal @ d
    n = g.num_cells
    A = np.bincount(owner, np.where(dot > 0.0, g.area * dot, 0.0), n)
    e = np.flatnonzero((kind == 0) & (dot < 0.0))
    target, source, w = owner[e], nb[e], g.area[e] * -dot[e]
    left = np.bincount(target, minlength=n)
    by = np.argsort(source, kind="stable")
    out_start = np.searchsorted(source[by], np.arange(n + 1))
    depth = np.zeros(n, np.int64)
    front, k, order, starts = np.flatnonzero(left == 0), 0, [], [0]
    while front.size:
        depth[front] = k
        order.append(front)
        starts.append(starts[-1] + front.size)
        lo, hi = out_start[front], out_start[front + 1]
        at = np.repeat(lo - np.concatenate(([0], np.cumsum(hi - lo)[:-1])), hi - lo) + np.arange((hi - lo).sum())
        down = target[by[at]]
        np.subtract.at(left, down, 1)
        down = np.unique(down)
        front, k = down[left[down] == 0], k + 1
    rank = np.argsort(depth[target], kind="stable")
    edge_starts = np.searchsorted(depth[target][rank], np.arange(len(starts)))
    p = np.flatnonzero((kind == 1) & (dot < 0.0))
    return (np.concatenate(order), starts, target[rank], source[rank], w[rank], edge_starts, A, owner[p], nb[p],
            g.area[p] * -dot[p])


CM3 = 1e-6
ERG = 1e-7
SIGMA = 2.9580524545305314e-18 * 1e-4
PROTON = 1.67262192369e-27


def absorbed_not(rho, x, size):
    return np.exp(-(rho / PROTON * (1.0 - x)) * SIGMA * size)


class Gas:
    """Hydrogen: the Rosdahl et al. (2015) rates and the semi-implicit sub-stepped update, on arrays of cells."""

    EV = 1.602176634e-19
    PHOTON = 18.028356312818811 * EV
    RYDBERG = 13.65693 * EV
    KB = 1.380649e-23
    FLOOR = 1e-10

    def __init__(self, rho, vol, size, rate):
        self.rho, self.vol, self.size, self.rate = rho, vol, size, rate
        self.nh = rho / PROTON

    def take(self, at):
        return Gas(self.rho[at], self.vol[at], self.size[at], self.rate[at])

    def newly_ionized(self, x, dt):
        return dt * self.rate * (1.0 - np.exp(-self.nh * (1.0 - x) * SIGMA * self.size))

    # the fits, each as its value and the derivative of its logarithm

    @staticmethod
    def collision(T):
        s = np.sqrt(T / 1e5)
        return np.sqrt(T) / (1.0 + s) * np.exp(-157809.1 / T), 0.5 / T - 0.5 * s / (T * (1.0 + s)) + 157809.1 / T ** 2

    @staticmethod
    def recombination(T):
        l = 315614.0 / T
        q = (l / 2.74) ** 0.407
        return 2.753e-14 * CM3 * l ** 1.5 / (1.0 + q) ** 2.242, -(1.5 - 2.242 * 0.407 * q / (1.0 + q)) / T

    @staticmethod
    def recombination_cooling(T):
        l = 315614.0 / T
        q = (l / 2.25) ** 0.376
        v = 3.435e-30 * ERG * CM3 * T * l ** 1.97 / (1.0 + q) ** 3.72
        return v, (1.0 - 1.97 + 3.72 * 0.376 * q / (1.0 + q)) / T

    @staticmethod
    def excitation(T):
        s = np.sqrt(T / 1e5)
        return 7.5e-19 * ERG * CM3 / (1.0 + s) * np.exp(-118348.0 / T), 118348.0 / T ** 2 - 0.5 * s / (T * (1.0 + s))

    def alpha(self, T):
        return self.recombination(T)[0]

    def beta(self, T):
        return 5.85e-11 * CM3 * self.collision(T)[0]

    def cooling(self, x, T, slope=False):
        pick = (lambda f: f[0] * f[1]) if slope else (lambda f: f[0])
        ne, n0 = self.nh * x, self.nh * (1.0 - x)
        coll = pick(self.excitation(T)) + 1.27e-21 * ERG * CM3 * pick(self.collision(T))
        brems = 1.42e-27 * ERG * CM3 * (0.5 / np.sqrt(T) if slope else np.sqrt(T))
        compton = 1.017e-37 * ERG * 2.727 ** 4 * (1.0 if slope else T - 2.727)
        return coll * ne * n0 + pick(self.recombination_cooling(T)) * ne * ne + brems * ne * ne + compton * ne

    def steps(self, x, T, dt):
        """The temperature's change, and the ionised fraction's as a function of the new temperature."""
        k = (5.0 / 3.0 - 1.0) * PROTON / (self.rho * self.KB)
        mu = 1.0 / (x + 1.0)
        heat = self.newly_ionized(x, dt) / self.vol * (self.PHOTON - self.RYDBERG) / dt
        dT = k * mu * (heat - self.cooling(x, T)) * dt / (1.0 + k * mu * self.cooling(x, T, True) * dt)

        def dx(T):
            ne = self.nh * x
            al, dal = self.recombination(T)
            be = 5.85e-11 * CM3
            c, dc = self.collision(T)
            dal, be, dbe = al * dal, be * c, be * c * dc
            C = be * ne + self.newly_ionized(x, dt) / (self.nh * (1.0 - x) * self.vol) / dt
            Dr = al * ne
            dC, dD = self.nh * be - ne * T * mu * dbe, self.nh * al - ne * T * mu * dal
            J = dC - (C + Dr) - x * (dC + dD)
            return dt * (C - x * (C + Dr)) / (1.0 - J * dt)

        return dT, dx

    def advance(self, x, T, dt0, safety):
        """Each cell's step, halved where a value would change by more than `safety`, halves in order."""
        n = len(x)
        depth, used = np.zeros(n, np.int64), np.zeros(n)
        pending = np.zeros((n, 64), bool)
        floor_x, floor_T = x.copy(), T.copy()

        def clamp(x, T, at):
            return np.clip(x, floor_x[at], 1.0 - self.FLOOR), np.maximum(T, floor_T[at])

        live = np.arange(n)
        while live.size:
            x[live], T[live] = clamp(x[live], T[live], live)
            part, dt = self.take(live), dt0 / 2.0 ** depth[live]
            dT, dx = part.steps(x[live], T[live], dt)
            rel_T = np.fmin(np.abs(dT / T[live]), 2.0 ** 52)
            T1 = T[live] + dT
            with np.errstate(all="ignore"):
                d = dx(T1)
                rel_x = np.fmin(np.abs(d / x[live]), 2.0 ** 52)
            ok = (rel_T <= safety) & (rel_x <= safety)
            good, bad = live[ok], live[~ok]
            x[good], T[good] = clamp(x[good] + d[ok], T1[ok], good)
            with np.errstate(divide="ignore"):
                used[good] = np.minimum(dt[ok] * (safety / rel_T[ok]), dt[ok] * (safety / rel_x[ok]))
            depth[bad] += 1
            pending[bad, depth[bad]] = True
            left = pending[good].any(axis=1)
            again = good[left]
            depth[again] = 63 - np.argmax(pending[again][:, ::-1], axis=1)
            pending[again, depth[again]] = False
            live = np.concatenate((bad, again))
        return x, T, used
