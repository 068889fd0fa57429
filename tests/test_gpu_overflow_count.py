"""GPU tests of the overflow count (PBF_OPT_COUNT_OVERFLOW), which every
wavefront of the list build adds to one of several counters: their sum over
more wavefronts than counters, with particles that get a wavefront of their own
among them, against the oracle; and that every build starts from zero."""
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lane_lists", [False, True])
@pytest.mark.parametrize("clump", [300, 4000])
def test_sum_over_wavefronts(pbf, scenes, clump, lane_lists):
    n = 12000
    rng = np.random.default_rng(clump)
    centres = rng.uniform(0.3, 2.7, size=(n // clump, 3))
    pos = (centres[rng.integers(0, len(centres), n)] + rng.uniform(-0.08, 0.08, size=(n, 3))).astype(np.float32)
    apart = scenes.lattice((24, 25, 20), spacing=0.11)
    params = scenes.pbf_params((3.0, 3.0, 3.0), n, count_overflow=True)
    if lane_lists:
        params.options |= pbf.PBF_OPT_LANE_LISTS
    g = pbf.Particles(params)
    g.add(pos)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=max(1, min(16, os.cpu_count() or 1)))
    o.set_state(pos, pos, np.zeros_like(pos))
    o.pass_(O.FIND)
    assert o.counters()["overflow"] > 0
    for again in range(2):
        g.set_position_stars(pos)
        g.find_neighbors()
        st = g.stats()
        assert st["neighbor_overflow"] == o.counters()["overflow"]
        assert st["tile_listed"] <= n
        g.set_position_stars(apart)
        g.find_neighbors()
        st = g.stats()
        assert st["neighbor_overflow"] == 0
        assert st["tile_listed"] == (0 if lane_lists else n)
    g.close()
    o.close()
