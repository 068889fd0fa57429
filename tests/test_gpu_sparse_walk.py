"""GPU tests of the list build where few particles share a cell, which a lane
each then lists: at the slots that a wavefront takes (4, 8, 16 and 32) and the
densities at which it changes over, with crowded cells next to lone particles,
particles that have left the grid or lost their position, short and long lists
and parts of the particles asked for.  Against the per-lane walk
(PBF_OPT_LANE_LISTS) and, in the smaller scenes, the oracle; all bit for bit."""
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def _lists(pbf, p, pos, lane, steps, spans=None):
    q = pbf.Params.from_buffer_copy(p)
    q.options |= pbf.PBF_OPT_LANE_LISTS if lane else 0
    g = pbf.Particles(q)
    g.add(pos)
    g.find_neighbors(*([] if spans is None else [pbf.span(*s) for s in spans]))
    lists, counts = g.neighbor_lists()
    over = g.stats()["neighbor_overflow"]
    if steps:
        g.step(steps)
    x = g.positions()
    g.close()
    mask = np.arange(lists.shape[1])[None, :] < counts[:, None]
    return np.where(mask, lists, 0), counts, over, x


def _compare(pbf, p, pos, steps=0, spans=None):
    a, b = (_lists(pbf, p, pos, lane, steps, spans) for lane in (False, True))
    assert np.array_equal(a[1], b[1])
    assert np.array_equal(a[0], b[0])
    assert a[2] == b[2]
    assert np.array_equal(a[3], b[3], equal_nan=True)
    return a


def _oracle(p, pos, got):
    o = O.Oracle(O.params_from_pbf(p), mode=O.JACOBI, threads=max(1, min(16, os.cpu_count() or 1)))
    o.set_state(pos, pos, np.zeros_like(pos))
    o.pass_(O.FIND)
    nb = o.neighbors()
    assert np.array_equal(got[1], nb["counts"])
    mask = np.arange(got[0].shape[1])[None, :] < got[1][:, None]
    assert np.array_equal(got[0], np.where(mask, nb["lists"], 0))
    o.close()


def _uniform(n, per_cell, seed=0):
    side = max(0.4, (n / per_cell) ** (1 / 3) * 0.12)
    return np.random.default_rng(seed + n).uniform(0.0, side, size=(n, 3)).astype(np.float32), side


@pytest.mark.parametrize("per_cell", [0.05, 0.9, 1.1, 1.9, 2.8, 3.5])
@pytest.mark.parametrize("n", [3, 9001, 20011, 140009, 530021])
def test_densities(pbf, scenes, n, per_cell):
    """Random points and three steps, the later ones over skin lists."""
    pos, side = _uniform(n, per_cell)
    p = scenes.pbf_params((side,) * 3, n, count_overflow=n % 2 == 0)
    got = _compare(pbf, p, pos, steps=3)
    if n < 30000:
        _oracle(p, pos, got)


@pytest.mark.parametrize("count_overflow", [False, True])
@pytest.mark.parametrize("cap", [1, 7, 60, 128])
@pytest.mark.parametrize("crowd", [100, 256, 257, 900])
def test_next_to_a_crowd(pbf, scenes, crowd, cap, count_overflow):
    """Lone particles among them crowds of one cell each: more candidates than
    a lane looks through, and lists that are full."""
    pos, side = _uniform(20000, 0.3)
    rng = np.random.default_rng(crowd)
    at = 0
    for centre in rng.uniform(0.5, side - 0.5, size=(6, 3)):
        pos[at:at + crowd] = centre + rng.uniform(0.0, 0.05, size=(crowd, 3))
        at += crowd
    pos = pos[rng.permutation(len(pos))]
    p = scenes.pbf_params((side,) * 3, len(pos), cap=cap, count_overflow=count_overflow)
    _oracle(p, pos, _compare(pbf, p, pos))


@pytest.mark.parametrize("n", [20000, 140000])
def test_particles_outside_the_grid(pbf, scenes, n):
    """Positions far off, infinite and lost, whole wavefronts of them and single ones."""
    pos, side = _uniform(n, 0.5)
    rng = np.random.default_rng(1)
    pos[: n // 4] += np.float32(1000.0)
    pos[n // 4: n // 3] = np.nan
    pos[rng.integers(0, n, 50)] = np.float32(np.inf)
    pos[rng.integers(0, n, 50), 1] = np.float32(-np.inf)
    pos[rng.integers(0, n, 50), 2] = np.nan
    p = scenes.pbf_params((side,) * 3, n, count_overflow=True)
    got = _compare(pbf, p, pos)
    lost = ~np.isfinite(pos).all(axis=1)
    assert not got[1][lost].any()


@pytest.mark.parametrize("spans", [((0, 20000), (0, 1)), ((0, 20000), (63, 12345)), ((0, 15000), (0, 20000)),
                                   ((0, 15000), (10000, 20000))])
def test_parts(pbf, scenes, spans):
    pos, side = _uniform(20000, 0.7)
    p = scenes.pbf_params((side,) * 3, len(pos))
    _compare(pbf, p, pos, spans=spans)


def test_batched(pbf, scenes):
    """Sparse scenes of different sizes in one context."""
    rng = np.random.default_rng(4)
    boxes = rng.uniform(2.0, 4.0, size=(12, 3)).astype(np.float32)
    n = 2500
    p = scenes.pbf_params(tuple(boxes[0]), n * len(boxes), count_overflow=True)
    out = []
    for lane in (0, pbf.PBF_OPT_LANE_LISTS):
        q = pbf.Params.from_buffer_copy(p)
        q.options |= lane
        g = pbf.Particles(q, boxes=boxes)
        for s, box in enumerate(boxes):
            x = (np.random.default_rng(s).uniform(0.0, 1.0, size=(n, 3)) * box).astype(np.float32)
            x[: s] += np.float32(50.0)
            g.add_to_scene(s, x)
        g.find_neighbors()
        lists, counts = g.neighbor_lists()
        mask = np.arange(lists.shape[1])[None, :] < counts[:, None]
        g.step(3)
        out.append((np.where(mask, lists, 0), counts, g.positions(), g.velocities()))
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
