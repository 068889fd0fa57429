"""GPU tests of the list builder's cell walk at the sizes where it changes: the
slots a wavefront takes (4, 8, 16 or 32), the 256 candidates of a chunk, the
eight particles of a group, the largest list of its two row lengths, and the
candidates above which a wavefront takes each particle by itself.  Lists,
counts and the overflow count against the per-lane walk (PBF_OPT_LANE_LISTS),
and the oracle where the grid is narrow; all bit for bit."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def _compare(pbf, p, pos, what, steps=0):
    out = []
    for lane in (0, pbf.PBF_OPT_LANE_LISTS):
        q = pbf.Params.from_buffer_copy(p)
        q.options |= lane
        g = pbf.Particles(q)
        g.add(pos, pos, np.zeros_like(pos))
        g.find_neighbors()
        lists, counts = g.neighbor_lists()
        over = g.stats()["neighbor_overflow"]
        if steps:
            g.step(steps)
        out.append((lists, counts, over, g.positions()))
        g.close()
    (la, ca, oa, xa), (lb, cb, ob, xb) = out
    assert np.array_equal(ca, cb), what + ": counts"
    mask = np.arange(la.shape[1])[None, :] < ca[:, None]
    assert np.array_equal(np.where(mask, la, 0), np.where(mask, lb, 0)), what + ": lists"
    assert oa == ob, what + ": overflow"
    assert np.array_equal(xa, xb), what + ": positions after the steps"
    return np.where(mask, la, 0), ca


@pytest.mark.parametrize("n", [1, 3, 13, 16384, 16385, 131072, 131073, 524288, 524293])
def test_sizes(pbf, scenes, n):
    """Random points (cells of 0 to some 30 particles), and three steps, the
    later ones over skin lists."""
    side = max(0.2, (n / 8000.0) ** (1 / 3))
    pos = np.random.default_rng(n).uniform(0.02, side, size=(n, 3)).astype(np.float32)
    p = scenes.pbf_params((side + 0.1,) * 3, n, count_overflow=True)
    _compare(pbf, p, pos, f"{n} particles", steps=3)


@pytest.mark.parametrize("count_overflow", [False, True])
@pytest.mark.parametrize("cap", [1, 60, 64, 65, 128])
@pytest.mark.parametrize("k", [1, 2, 7, 8, 9, 64, 65, 129, 255, 256, 257, 513, 1536, 1537, 3072, 3073])
def test_streams(pbf, scenes, k, cap, count_overflow):
    """k particles in one cell (k candidates each, all accepted: the cell is
    smaller than the spacing), next to a cell of three."""
    rng = np.random.default_rng(k)
    pos = np.concatenate([rng.uniform(0.40, 0.44, size=(k, 3)), rng.uniform(0.70, 0.74, size=(3, 3))]).astype(np.float32)
    p = scenes.pbf_params((1.0, 1.0, 1.0), pos.shape[0], cap=cap, count_overflow=count_overflow)
    _compare(pbf, p, pos, f"{k} in a cell, cap {cap}")


@pytest.mark.parametrize("far", [40, 1600, 1800, 3000])
def test_hand_on(pbf, scenes, far):
    """More than 3,072 candidates of which `far` come before the near ones and
    are out of reach: lists not full when the walk's 1,536 are tested go on to
    a wavefront of their own."""
    rng = np.random.default_rng(far)
    s = 0.12
    lo = np.array([2.0 * s, 3.05 * s, 3.05 * s])
    pos = np.concatenate([lo + rng.uniform(0.0, 0.1 * s, size=(far, 3)), [[3.9 * s, 3.9 * s, 3.9 * s]],
                          [3.9 * s, 3.9 * s, 3.9 * s] + rng.uniform(-0.05, 0.05, size=(20, 3)) * s,
                          [4.95 * s, 3.9 * s, 3.9 * s] + rng.uniform(0.0, 0.04, size=(3200, 3)) * s]).astype(np.float32)
    p = scenes.pbf_params((1.0, 1.0, 1.0), pos.shape[0])
    _compare(pbf, p, pos, f"{far} far candidates first")


@pytest.mark.parametrize("box", [(0.1, 0.1, 1.0), (0.1, 1.0, 1.0), (1.0, 0.1, 0.3), (0.2, 0.2, 0.2)])
@pytest.mark.parametrize("cap", [60, 128])
def test_narrow_grids(pbf, scenes, box, cap):
    """Grids of three or four cells an axis, whose walks wrap from row to row."""
    n = 400
    pos = (np.random.default_rng(5).uniform(0.0, 1.0, size=(n, 3)) * np.array(box)).astype(np.float32)
    p = scenes.pbf_params(box, n, cap=cap, count_overflow=True)
    lists, counts = _compare(pbf, p, pos, f"box {box}")
    o = O.Oracle(O.params_from_pbf(p), mode=O.JACOBI, threads=1)
    o.set_state(pos, pos, np.zeros_like(pos))
    o.pass_(O.FIND)
    nb = o.neighbors()
    assert np.array_equal(counts, nb["counts"])
    mask = np.arange(cap)[None, :] < counts[:, None]
    assert np.array_equal(lists, np.where(mask, nb["lists"], 0))
    o.close()
