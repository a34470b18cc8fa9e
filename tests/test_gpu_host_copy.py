"""Copies between host arrays and the device at the sizes where their route changes: up to one chunk (1 MiB,
the runtime's copy), one byte range past it, and more chunks than there are pinned buffers."""
import ctypes as C
import threading

import numpy as np
import pytest

from lambda_amd import abi, gpu, scene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = gpu.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("w,h", [(1, 1), (209, 209), (256, 171), (210, 210), (1000, 701), (1021, 1531)])
def test_film_round_trip(dev, w, h):
    rng = np.random.default_rng(w * h)
    rgb = rng.random((h, w, 3))
    cnt = rng.integers(0, 9, (h, w)).astype(np.uint32)
    f = gpu.Film(dev, w, h)
    f.write(rgb, cnt)
    r, c = f.read()
    np.testing.assert_array_equal(r, rgb)
    np.testing.assert_array_equal(c, cnt)
    f.close()


def test_two_devices_copy_at_once(dev):
    """Two device objects on one GPU, each with its own buffers and threads, read from two host threads."""
    other = gpu.Device(0)
    rng = np.random.default_rng(1)
    films, want, got = [], [], [None, None]
    for d in (dev, other):
        f = gpu.Film(d, 800, 600)
        a = rng.random((600, 800, 3))
        f.write(a)
        films.append(f)
        want.append(a)

    def read(k):
        got[k] = [films[k].read()[0] for _ in range(4)]
    ts = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in range(2):
        for a in got[k]:
            np.testing.assert_array_equal(a, want[k])
    for f in films:
        f.close()
    other.close()


@pytest.mark.parametrize("n", [1, 32768, 32769, 600001])
def test_ray_batches(dev, n):
    """A batch's answers are those of its rays in small batches."""
    s = gpu.Scene(dev)
    keep = scene.cornell_box().push(s, abi.LIGHTS_TREE)
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = rng.uniform(-0.9, 0.9, size=(n, 3))
    rays = np.concatenate([o, np.zeros((n, 1)), d, np.full((n, 1), np.inf)], axis=1).astype(np.float32)
    hits, occ = s.intersect(rays), s.occluded(rays)
    for a in {0, max(0, n // 2 - 500), max(0, n - 1000)}:
        np.testing.assert_array_equal(hits[a:a + 1000], s.intersect(rays[a:a + 1000]))
        np.testing.assert_array_equal(occ[a:a + 1000], s.occluded(rays[a:a + 1000]))
    del keep
    s.close()


@pytest.mark.parametrize("w,h", [(209, 209), (210, 210), (1021, 1531)])
def test_film_round_trip_through_page_locked_arrays(dev, w, h):
    n = 3 * w * h
    L = gpu.lib()  # its handle gives the HIP runtime's own functions too
    L.hipHostMalloc.argtypes = [C.c_void_p, C.c_size_t, C.c_uint]
    L.hipHostFree.argtypes = [C.c_void_p]
    p = C.c_void_p()
    assert L.hipHostMalloc(C.byref(p), 8 * (2 * n + 5), 0) == 0
    mem = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (2 * n + 5,))
    up, down = mem[5:5 + n], mem[5 + n:]
    up[:] = np.random.default_rng(n).random(n)
    down[:] = 0.0
    f = gpu.Film(dev, w, h)
    cnt = np.ones((h, w), dtype=np.uint32)
    assert L.lgpu_film_write(f.h, up.ctypes.data_as(C.c_void_p), cnt.ctypes.data_as(C.c_void_p)) == abi.OK
    assert L.lgpu_film_read(f.h, down.ctypes.data_as(C.c_void_p), None) == abi.OK
    np.testing.assert_array_equal(down, up)
    np.testing.assert_array_equal(f.read()[0].reshape(-1), up)
    f.close()
    L.hipHostFree(p)
