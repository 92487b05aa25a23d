"""GPU: the direction sweeps' tiles where their layout has edges. Bitwise equal
to the grouped replay (X, I, fields) on grids made by hand:

  hub     a cell with 4, 13, 14, 21 or 115 upwind faces (entries in the planes,
          one more, and more extra entries than a wave has lanes) behind 200
          level sets that hold more tasks than the LDS ring, so that its upwind
          values are far ones (more than 64 for the largest);
  slab    4 x m x m cells along an axis: level sets wider than the ring
          (m = 190: every upwind value is a far one) and between a quarter of
          it and the whole (m = 110), which wait for the level set before;
  tiny    1 to 65 cells in a row: fewer tiles than waves, partial tiles.
"""

import numpy as np
import pytest

from oracle.oracle import OracleSweep
from subsweep_amd import Sweep, SweepParameters
from subsweep_amd.grid import Grid

pytestmark = pytest.mark.gpu

MYR = 3.15576e13


def _grid(n, i, j, normal, area, boundary=()):
    """Cells 0..n-1 with local faces i -> j (and their mirrors) and boundary
    faces (cell, normal)."""
    b = np.array([c for c, _ in boundary], np.int64)
    bn = np.array([v for _, v in boundary], np.float64).reshape(-1, 3)
    owner = np.concatenate([i, j, b])
    nbr = np.concatenate([j, i, np.zeros(len(b), np.int64)])
    nrm = np.concatenate([normal, -normal, bn])
    ar = np.concatenate([area, area, np.ones(len(b))])
    kind = np.concatenate([np.zeros(2 * len(i), np.uint8), np.full(len(b), 2, np.uint8)])
    o = np.argsort(owner, kind="stable")
    off = np.concatenate([[0], np.cumsum(np.bincount(owner, minlength=n))])
    rng = np.random.default_rng(n)
    return Grid(off, nbr[o].astype(np.int32), kind[o], ar[o] * 1e40, nrm[o], rng.uniform(1.0, 2.0, n) * 1e60,
                np.full(n, 1e20), points=rng.random((n, 3)))


def _unit(v):
    return v / np.linalg.norm(v, axis=1)[:, None]


def _hub(up):
    rng = np.random.default_rng(up)
    chains, length = 181, 200  # 36200 tasks before the hub's level set
    first = 1 + up
    col = first + np.arange(chains)[:, None] * length + np.arange(length)
    i = np.concatenate([np.arange(1, 1 + up), col[:, :-1].ravel(), col[:1, -1]])
    j = np.concatenate([np.zeros(up, np.int64), col[:, 1:].ravel(), [0]])
    normal = _unit(np.column_stack([np.ones(len(i)), rng.uniform(-0.5, 0.5, (len(i), 2))]))
    n = first + chains * length
    bd = [(0, (1.0, 0.0, 0.0))] + [(int(c), (0.0, 1.0, 0.0)) for c in col[:, 0]]
    return _grid(n, i, j, normal, rng.uniform(0.5, 2.0, len(i)), bd), [[1.0, 0.0, 0.0], [-1.0, 0.1, 0.0]]


def _slab(m):
    c = np.arange(4 * m * m).reshape(4, m, m)
    pairs = [(c[:-1].ravel(), c[1:].ravel(), (1.0, 0.0, 0.0)), (c[:, :-1].ravel(), c[:, 1:].ravel(), (0.0, 1.0, 0.0)),
             (c[:, :, :-1].ravel(), c[:, :, 1:].ravel(), (0.0, 0.0, 1.0))]
    i, j = (np.concatenate([p[k] for p in pairs]) for k in (0, 1))
    normal = np.concatenate([np.tile(p[2], (len(p[0]), 1)) for p in pairs])
    return _grid(c.size, i, j, normal, np.ones(len(i))), [[1.0, 0.0, 0.0], [-1.0, 0.02, 0.03], [0.0, 1.0, 0.0],
                                                          [0.6, 0.7, -0.4]]


def _tiny(n):
    i = np.arange(n - 1)
    normal = _unit(np.column_stack([np.ones(n - 1), np.sin(i), np.cos(i)]))
    return _grid(n, i, i + 1, normal, 1.0 + i, [(n - 1, (1.0, 0.0, 0.0))]), [[1.0, 0.2, 0.1], [0.1, 1.0, 0.3]]


CASES = {f"hub{k}": lambda k=k: _hub(k) for k in (4, 13, 14, 21, 115)}
CASES.update({f"slab{m}": lambda m=m: _slab(m) for m in (110, 190)})
CASES.update({f"tiny{k}": lambda k=k: _tiny(k) for k in (1, 2, 64, 65)})


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", list(CASES))
def test_tiles_bitwise_equal_grouped(name, precision, hip_available):
    grid, dirs = CASES[name]()
    n = grid.num_cells
    rng = np.random.default_rng(1)
    src = np.where(rng.random(n) < 0.2, 10.0 ** rng.uniform(48, 50, n), 0.0)
    src[: min(n, 120)] = 1e49
    state = (1e-27 * np.exp(rng.standard_normal(n)), np.full(n, 1e-10), np.full(n, 1e4), src)
    p = SweepParameters(directions=dirs, num_timestep_levels=3, max_timestep=1e-3 * MYR,
                        transport_precision=precision)
    with Sweep(p, grid, *state) as a, Sweep(p, grid, *state, direction_sweeps=True) as b:
        assert b.info().direction_sweeps == 1
        for step in range(4):
            assert a.run_sweeps() == b.run_sweeps()
            for u, v in zip(a.transport_state(), b.transport_state()):
                assert np.array_equal(u.view(np.uint8), v.view(np.uint8)), f"step {step}"
            ra, rb = a.results(), b.results()
            assert np.array_equal(ra.ionized_hydrogen_fraction, rb.ionized_hydrogen_fraction)
            assert np.array_equal(ra.photon_rate, rb.photon_rate) and np.array_equal(ra.level, rb.level)
        assert np.count_nonzero(a.transport_state()[1]) > n // 2 or n == 1


@pytest.mark.parametrize("name", ["tiny1", "tiny65", "hub115", "slab110", "slab190"])
def test_level_sets_equal_the_oracles(name, hip_available):
    # counters in LDS and (slab190: 144400 cells) in memory, level sets that
    # fit in the queues and ones that go on in memory
    grid, dirs = CASES[name]()
    n = grid.num_cells
    state = (np.full(n, 1e-27), np.full(n, 1e-10), np.full(n, 1e4), np.full(n, 1e48))
    p = SweepParameters(directions=dirs, num_timestep_levels=2, max_timestep=1e-3 * MYR)
    o = OracleSweep(p, grid, *state)
    with Sweep(p, grid, *state) as s:
        for lvl in range(2):
            assert np.array_equal(s.counts(lvl), o.counts(lvl)) and np.array_equal(s.levelsets(lvl), o.levelsets(lvl))
    o.close()
