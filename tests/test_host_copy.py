"""Copies between host arrays and the device: which route they take, and what they give back. Run on the CPU
(tests/host_hip.py)."""
from tests.host_hip import host_hip  # noqa: F401


def test_every_pinned_buffer_is_used(host_hip):
    """A copy of many chunks goes through all of the pinned memory that the device object holds."""
    host_hip("""
f = gpu.Film(dev, 2048, 1500)
before = H.host_hip_pinned()
for _ in range(4): f.read()
held = H.host_hip_pinned() - before
assert held == 12 * MB, held
""")


def test_small_copies_wait_for_no_other_thread(host_hip):
    """A read of two chunks (1.5 MiB) is done by the calling thread; longer ones give what was written,
    whichever thread takes which chunk."""
    host_hip("""
f = gpu.Film(dev, 256, 256)
a = np.random.default_rng(0).random((256, 256, 3))
f.write(a)
copies()
me = threading.get_native_id()
for _ in range(20):
    got, cnt = f.read()
    assert (got == a).all()
    big = [c for c in copies() if c[1] > 512 * 1024]
    assert big and all(c[3] == me for c in big), big
for w, h in ((256, 300), (512, 341), (1021, 1531)):
    f = gpu.Film(dev, w, h)
    a = np.random.default_rng(1).random((h, w, 3))
    f.write(a)
    for _ in range(20):
        assert (f.read()[0] == a).all()
""")


def test_page_locked_and_device_memory_is_copied_directly(host_hip):
    """A page-locked array, or device memory in the place of a host array, takes one copy of the whole
    range, in both directions and from any place inside the allocation; an ordinary array goes by chunks."""
    host_hip("""
H.hipHostMalloc.argtypes = [C.c_void_p, C.c_size_t, C.c_uint]
H.hipMalloc.argtypes = [C.c_void_p, C.c_size_t]
L = gpu.lib()
w, h = 1600, 1100
n = 24 * w * h
f = gpu.Film(dev, w, h)
a = np.random.default_rng(3).random((h, w, 3))
for kind in ("pinned", "device"):
    p = C.c_void_p()
    assert (H.hipHostMalloc(C.byref(p), n + 4096, 0) if kind == "pinned" else H.hipMalloc(C.byref(p), n + 4096)) == 0
    at = p.value + 264
    C.memmove(at, a.ctypes.data, n)
    cnt = np.ones((h, w), dtype=np.uint32)
    copies()
    assert L.lgpu_film_write(f.h, at, cnt.ctypes.data) == 0
    assert [c for c in copies() if c[0] == at and c[1] == n and c[2] == 1], kind
    C.memset(at, 0, n)
    assert L.lgpu_film_read(f.h, at, None) == 0
    c = copies()
    assert len(c) == 1 and c[0][0] == at and c[0][1] == n, (kind, c)
    assert C.string_at(at, n) == a.tobytes()
copies()
f.read()
assert sum(c[1] == MB for c in copies()) == n // MB + 4 * w * h // MB
""")
