"""GPU tests of the stable radix sort at the edges of its plan: the tile sizes
(1,024 keys up to 2^18, 4,096 above), one tile and one group more or less,
odd digit widths, and the sizes past 2,048 tiles where the groups are turned
into prefixes first; and of the list build around the scene size below which
no particle can need the wavefront builder."""
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

SIZES = [(2, 1), (1023, 9), (1025, 32), (65 * 1024 + 1, 17), (1 << 18, 16), ((1 << 18) + 1, 19), (290_001, 25),
         (1_000_003, 20), (8_388_608, 22), (8_388_609, 23), (9_000_001, 11)]


@pytest.mark.parametrize("n,bits", SIZES)
def test_sort_at_the_plan_edges(pbf, n, bits):
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << bits, size=n, dtype=np.uint64).astype(np.uint32)
    keys[::3] = keys[0]  # long runs of one key: stability shows
    vals = rng.permutation(n).astype(np.uint32)
    sk, sv = pbf.sort_by_key_u32(keys, vals, bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(sk, keys[order])
    assert np.array_equal(sv, vals[order])


@pytest.mark.parametrize("count_overflow", [False, True])
@pytest.mark.parametrize("n", [700, 768, 769, 1024, 1025, 1600])
def test_crowded_scene_around_the_lane_limit(pbf, scenes, n, count_overflow):
    """All particles in a few cells: with 768 (overflow counted) or 1,024
    candidates the lanes list every particle, above the wavefront builder
    takes some; lists, counts and overflow equal the oracle's either way."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.3, 0.55, (n, 3)).astype(np.float32)
    params = scenes.pbf_params((1.2, 0.8, 0.8), n, cap=60, count_overflow=count_overflow)
    g = pbf.Particles(params)
    g.add(pos)
    g.find_neighbors()
    lists, counts = g.neighbor_lists()
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=max(1, min(16, os.cpu_count() or 1)))
    o.set_state(pos, pos, np.zeros_like(pos))
    o.pass_(O.FIND)
    nb = o.neighbors()
    assert np.array_equal(counts, nb["counts"])
    for p in range(n):
        assert np.array_equal(lists[p, :counts[p]], nb["lists"][p, :counts[p]]), p
    if count_overflow:
        assert g.stats()["neighbor_overflow"] == o.counters()["overflow"]
    g.close()


@pytest.mark.parametrize("bits", [1, 7, 8, 9, 17, 24, 32])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1023, 1024, 1025, 2049, 4095, 4096, 4097])
def test_sort_around_one_block(pbf, n, bits):
    """Up to 1,024 and 4,096 keys are sorted by one block, in LDS: stable, and
    equal to the sort of numpy, with one to four passes."""
    rng = np.random.default_rng(100 * n + bits)
    keys = rng.integers(0, 1 << (min(bits, 6) if n % 2 else bits), size=n, dtype=np.uint64).astype(np.uint32)
    vals = rng.permutation(n).astype(np.uint32)
    k, v = pbf.sort_by_key_u32(keys, vals, bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k, keys[order])
    assert np.array_equal(v, vals[order])
