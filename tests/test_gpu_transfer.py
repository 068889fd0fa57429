"""GPU tests of the copies between ordinary memory and the device at the sizes
where their route changes: kernels on pinned memory up to 64 KB, one chunk up
to 2 MB, one thread up to 8 MB, two up to 32 MB, four above; and device
pointers.  Arrays must come back as they were set, in the particles' order."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(pbf, scenes, n, seed):
    side = max(0.3, (n / 8000.0) ** (1 / 3))
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.02, side, size=(n, 3)).astype(np.float32)
    p = pbf.Particles(scenes.pbf_params((side + 0.1,) * 3, n))
    p.add(pos, pos, np.zeros_like(pos))
    p.find_neighbors()  # particles now lie in cell order
    return p, rng


# bytes / 12 and / 4 at each limit, one particle less and more
@pytest.mark.parametrize("n", [1, 2, 5461, 5462, 16384, 16385, 174762, 174763, 524289, 262145, 699050, 699051, 2796202,
                               2796203])
def test_arrays_come_back(pbf, scenes, n):
    p, rng = _context(pbf, scenes, n, n)
    for k in range(2):  # (the second pass over used staging memory)
        x = rng.standard_normal((n, 3)).astype(np.float32)
        v = rng.standard_normal((n, 3)).astype(np.float32)
        rho = rng.standard_normal(n).astype(np.float32)
        p.set_positions(x)
        p.set_velocities(v)
        p.set_densities(rho)
        assert np.array_equal(p.velocities(), v)
        assert np.array_equal(p.densities(), rho)
        assert np.array_equal(p.positions(), x)
    p.close()


@pytest.mark.parametrize("n", [100, 100000])
def test_device_pointers(pbf, scenes, n):
    p, rng = _context(pbf, scenes, n, 3)
    x = rng.standard_normal((n, 3)).astype(np.float32)
    back = np.zeros_like(x)
    L = pbf.lib()
    fp, vp = ctypes.POINTER(ctypes.c_float), ctypes.c_void_p
    given, got = vp(), vp()
    for d in (given, got):
        assert L.pbf_device_alloc(x.nbytes, ctypes.byref(d)) == 0
    assert L.pbf_memcpy_to_device(given, x.ctypes.data_as(vp), x.nbytes) == 0
    assert L.pbf_set_positions(p._ctx, ctypes.cast(given, fp)) == 0
    assert np.array_equal(p.positions(), x)
    assert L.pbf_get_positions(p._ctx, ctypes.cast(got, fp)) == 0
    assert L.pbf_memcpy_to_host(back.ctypes.data_as(vp), got, x.nbytes) == 0
    assert np.array_equal(back, x)
    for d in (given, got):
        L.pbf_device_free(d)
    p.close()


@pytest.mark.parametrize("count", [1, 17, 32767, 32768, 32769, 150000])
def test_predict_in_blocks_of_rows(pbf, count):
    """Rows past one launch's 32,768 give what they give alone."""
    m = pbf.WarmModel(count)
    m.init(5)
    f = np.random.default_rng(2).uniform(-1, 1, size=(count, 8)).astype(np.float32)
    whole = m.predict(f)
    for first in {0, max(0, count - 40), min(32752, max(0, count - 40))}:
        assert np.array_equal(whole[first:first + 40], m.predict(f[first:first + 40]))
