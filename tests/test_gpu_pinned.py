"""GPU tests of calls on arrays in pinned host memory: the library tells the
three kinds of memory apart (pinned and device memory are copied as they are,
without the staging memory), and arrays come back as they were set at the sizes
where the route changes."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAGEABLE, PINNED, DEVICE = 0, 1, 2


class _Pinned:
    """An array in memory that the runtime has allocated pinned."""

    def __init__(self, pbf, shape):
        pbf.lib()
        self.hip = ctypes.CDLL("libamdhip64.so.7")  # (the one that the library has loaded)
        self.ptr = ctypes.c_void_p()
        nbytes = 4 * int(np.prod(shape))
        assert self.hip.hipHostMalloc(ctypes.byref(self.ptr), ctypes.c_size_t(nbytes), ctypes.c_uint(0)) == 0
        self.array = np.frombuffer((ctypes.c_char * nbytes).from_address(self.ptr.value), np.float32).reshape(shape)

    def free(self):
        self.array = None
        self.hip.hipHostFree(self.ptr)


def _fp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def test_kinds_of_memory(pbf):
    memory_of = getattr(pbf.lib(), "_ZN3pbf9memory_ofEPKv")
    memory_of.argtypes, memory_of.restype = [ctypes.c_void_p], ctypes.c_int
    a = np.zeros(1000, np.float32)
    h = _Pinned(pbf, 1000)
    d = pbf.DeviceBuffer(4000)
    assert memory_of(a.ctypes.data) == PAGEABLE
    assert memory_of(h.ptr) == PINNED and memory_of(h.ptr.value + 1996) == PINNED
    assert memory_of(d.ptr) == DEVICE and memory_of(d.ptr.value + 1996) == DEVICE
    d.free()
    h.free()


@pytest.mark.parametrize("n", [1, 2730, 2731, 5461, 5462, 174763, 699051, 2796203])
def test_pinned_arrays_come_back(pbf, scenes, n):
    side = max(0.3, (n / 8000.0) ** (1 / 3))
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.02, side, size=(n, 3)).astype(np.float32)
    given, got = _Pinned(pbf, (n, 3)), _Pinned(pbf, (n, 3))
    given.array[:] = pos
    L = pbf.lib()
    p = pbf.Particles(scenes.pbf_params((side + 0.1,) * 3, n))
    assert L.pbf_add(p._ctx, _fp(given.array), _fp(pos), _fp(given.array), n) == 0  # pinned and not, in turn
    assert np.array_equal(p.positions(), pos)
    assert np.array_equal(p.velocities(), pos)
    p.find_neighbors()  # particles now lie in cell order
    v = rng.standard_normal((n, 3)).astype(np.float32)
    given.array[:] = v
    assert L.pbf_set_velocities(p._ctx, _fp(given.array)) == 0
    assert L.pbf_get_velocities(p._ctx, _fp(got.array)) == 0
    assert np.array_equal(got.array, v)
    assert L.pbf_set_densities(p._ctx, _fp(given.array)) == 0
    assert L.pbf_get_densities(p._ctx, _fp(got.array)) == 0
    assert np.array_equal(got.array.reshape(-1)[:n], v.reshape(-1)[:n])
    p.close()
    given.free()
    got.free()
