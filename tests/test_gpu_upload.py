"""GPU: grids whose upload has edges, against the oracle's fluxes: faces in one
chunk and in several (a single direction leaves little staging room), with and
without periodic cells, in the caller's and in Morton order; and the first
invalid face (in the internal order) is what the error names.

Bar: 1e-11 of the largest rate for the FP64 rates (sums over at most 6 faces
a cell in the same order; a few hundred cells in a row at 2^-52 each)."""

import dataclasses

import numpy as np
import pytest

from oracle.oracle import OracleSweep
from subsweep_amd import Sweep, SweepParameters
from subsweep_amd import _native as N
from subsweep_amd import grid as G
from subsweep_amd import workloads as W

pytestmark = pytest.mark.gpu

MYR = 3.15576e13


def _problem(n, periodic, directions):
    g = G.cartesian_grid(n, W.BOX, periodic)
    rng = np.random.default_rng(n)
    src = np.where(rng.random(g.num_cells) < 0.1, 1e48, 0.0)
    src[0] = 1e48
    gas = (W.RHO_MEAN * 10.0 ** rng.uniform(-3, 0, g.num_cells), np.full(g.num_cells, 1e-6),
           np.full(g.num_cells, 1e3), src)
    return SweepParameters(directions=directions, num_timestep_levels=2, max_timestep=1e-3 * MYR,
                           periodic=periodic), g, gas


@pytest.mark.parametrize("positions", [True, False])
@pytest.mark.parametrize("n,periodic,directions", [(1, False, 1), (2, True, 1), (24, True, 1), (24, False, 1),
                                                   (9, True, 16)])
def test_uploaded_grid_equals_the_oracles(n, periodic, directions, positions, hip_available):
    p, g, gas = _problem(n, periodic, directions)
    if not positions:
        g = dataclasses.replace(g, points=None)
    o = OracleSweep(p, g, *gas)
    with Sweep(p, g, *gas) as s:
        assert s.info().locality_order == (1 if positions and g.points is not None else 0)
        for lvl in range(2):
            assert np.array_equal(s.counts(lvl), o.counts(lvl)) and np.array_equal(s.levelsets(lvl), o.levelsets(lvl))
        for _ in range(2):
            assert s.run_sweeps() == o.run_sweeps()
        for a, b in zip(s.fluxes(), o.fluxes()):
            assert np.abs(a - b).max() <= 1e-11 * max(np.abs(b).max(), 1.0)
    o.close()


def test_first_invalid_face_is_named(hip_available):
    p, g, gas = _problem(24, True, 1)
    g = dataclasses.replace(g, points=None)
    for first, second, text in (((7, 3, None), (80000, None, -1), "face_kind"),
                                ((7, None, g.num_cells), (80000, 3, None), "out of range"),
                                ((82943, None, -1), (82943, 3, None), "face_kind")):
        kind, nbr = g.kind.copy(), g.neighbour.copy()
        for f, k, b in (first, second):
            if b is not None:
                nbr[f] = b
                kind[f] = 0
        for f, k, b in (first, second):
            if k is not None:
                kind[f] = k
        with pytest.raises(N.SweepError, match=text):
            Sweep(p, dataclasses.replace(g, kind=kind, neighbour=nbr), *gas)
