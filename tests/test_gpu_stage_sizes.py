"""GPU tests of transfers at the sizes that an object's staging memory holds
and just past them: the neighbour lists and cell bounds of small contexts (one
slot of staging memory), the samples of a warm-start model (two slots of
512 KB), and predictions past the rows that the model has a workspace for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 21, 100, 1000, 6000])
def test_lists_of_small_contexts(pbf, scenes, n):
    """Lists, counts and bounds, which are larger than a small context's
    staging memory, against the same particles in a large context."""
    pos = np.random.default_rng(n).uniform(0.02, 0.9, size=(n, 3)).astype(np.float32)
    out = []
    for capacity in (n, 2_000_000):
        p = pbf.Particles(scenes.pbf_params((1.0, 1.0, 1.0), capacity))
        p.add(pos)
        p.find_neighbors()
        out.append((*p.neighbor_lists(), *p.bin_bounds(), p.particle_ids(), p.bin_ids()))
        p.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("count", [1, 5, 16383, 16384, 16385, 32768, 32769, 131072, 131073, 262145])
def test_samples_arrive(pbf, count):
    """The gradient of one stored sample is that of the same sample alone, for
    the first and last samples of arrays of any size, stored in two calls."""
    rng = np.random.default_rng(count)
    f = rng.uniform(-1, 1, size=(count, 8)).astype(np.float32)
    t = rng.uniform(-1, 1, size=count).astype(np.float32)
    m, one = pbf.WarmModel(count + 3), pbf.WarmModel(1)
    m.init(7)
    one.init(7)
    m.add_samples(np.ones((3, 8), np.float32), np.ones(3, np.float32))
    m.add_samples(f, t)
    for i in {0, count // 2, max(0, 16384 - 1) % count, count - 1}:
        one.clear_samples()
        one.add_samples(f[i:i + 1], t[i:i + 1])
        g, loss = m.gradient(3 + i, 1)
        g1, loss1 = one.gradient(0, 1)
        assert loss == loss1 and np.array_equal(g, g1), i
    m.close()
    one.close()


@pytest.mark.parametrize("count", [32768, 65537, 524288, 524289, 600001])
def test_predict_past_the_workspace(pbf, count):
    """Every row equals its prediction in calls of 1,000 rows."""
    m = pbf.WarmModel(8)
    m.init(3)
    f = np.random.default_rng(1).uniform(-1, 1, size=(count, 8)).astype(np.float32)
    whole = m.predict(f)
    parts = np.concatenate([m.predict(f[i:i + 1000]) for i in range(0, count, 1000)])
    assert np.array_equal(whole, parts)
    m.close()
