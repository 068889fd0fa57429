"""GPU tests of the list build where walk cells repeat: x + i*s rounds into the
cell of x + (i-1)*s on a wall, so a particle there meets candidates twice an
axis and has more of them than the scene has particles.  At scene sizes on both
sides of those from which the wavefront builder runs, with both walks; lists,
counts, overflow and two steps against the oracle, bit for bit."""
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

WALL = np.float32(2.4)


def _cells(x, s):
    """The walk's three cells on an axis, in float (neighbors.h:110-111,177-179)."""
    x, s = np.float32(x), np.float32(s)
    return [int(np.floor(np.float32(np.float32(x + np.float32(i) * s) + s) / s)) for i in (-1, 0, 1)]


def _scene(n):
    """A few particles in the corner of three walls, the others in the far part
    of the corner's cell, out of reach of them: a corner particle has eight
    times the scene as candidates, and its list is not full after the budget of
    either walk."""
    rng = np.random.default_rng(n)
    near = min(max(4, n // 10), 14)
    pos = rng.uniform(2.281, 2.30, size=(n, 3)).astype(np.float32)
    pos[:near] = rng.uniform(2.36, 2.40, size=(near, 3)).astype(np.float32)
    pos[:3 * near // 4, 0] = WALL
    pos[:2 * near // 4, 1] = WALL
    pos[:max(2, near // 4), 2] = WALL
    return pos[rng.permutation(n)]


@pytest.mark.parametrize("lane_lists", [False, True])
@pytest.mark.parametrize("count_overflow", [False, True])
@pytest.mark.parametrize("budget", [64, 768])
@pytest.mark.parametrize("n", [40, 64, 65, 128, 129, 256, 257, 600, 768, 769, 1024, 1025, 1536, 1537, 3072, 3073])
def test_repeated_walk_cells(pbf, scenes, n, budget, count_overflow, lane_lists):
    pos = _scene(n)
    params = scenes.pbf_params((2.4, 2.4, 2.4), n, cap=60, count_overflow=count_overflow)
    if lane_lists:
        params.options |= pbf.PBF_OPT_LANE_LISTS
    w = _cells(WALL, params.neighbor_bin_spacing)
    assert w[0] == w[1]  # the wall's walk cells repeat
    g = pbf.Particles(params)
    g.set_tuning(heavy_budget=budget)
    g.add(pos)
    g.find_neighbors()
    lists, counts = g.neighbor_lists()
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=max(1, min(16, os.cpu_count() or 1)))
    o.set_state(pos, pos, np.zeros_like(pos))
    o.pass_(O.FIND)
    nb = o.neighbors()
    assert np.array_equal(counts, nb["counts"])
    mask = np.arange(60)[None, :] < counts[:, None]
    assert np.array_equal(np.where(mask, lists, 0), np.where(mask, nb["lists"], 0))
    if count_overflow:
        assert g.stats()["neighbor_overflow"] == o.counters()["overflow"]
    # (the second step walks the skin lists that the first one allows, if any)
    o.set_state(pos, pos, np.zeros_like(pos))
    for _ in range(2):
        g.step(1)
        o.step(1)
        assert np.array_equal(g.positions(), o.state()["x"].astype(np.float32))
    g.close()
    o.close()
