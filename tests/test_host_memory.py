"""Device memory that the library keeps between calls, and what a failed call gives back. Run on the CPU
(tests/host_hip.py) with a budget of device memory, so that allocations fail part way."""
from tests.host_hip import host_hip  # noqa: F401

GIB = 1 << 30

BATCH = """
GIB = 1 << 30
def job(side, spp, s, cap=0):
    f = gpu.Film(dev, side, side)
    return gpu.render_desc(s, f, scene.cornell_camera(side, side), 0, spp, max_bounces=4, estimator=abi.ESTIMATOR_CORRECTED,
                           capacity=cap), f
s = gpu.Scene(dev)
scene.cornell_box().push(s, abi.LIGHTS_TREE)
small, fs = job(64, 4, s)
large, fl = job(1024, 64, s)          # 2^26 paths, some 22 GiB
fits, ff = job(1024, 8, s)            # 2^23 paths, 2.8 GiB
"""


def test_failed_batch_gives_its_pool_back(host_hip):
    """A batch that runs out of device memory keeps nothing of its pool: what fits afterwards is what fitted
    before, a small batch and a render among it."""
    host_hip(BATCH + """
before = live()
H.host_hip_budget(before + 7 * GIB // 2)
try:
    gpu.render_batch([large], path_capacity=1 << 26)
    raise SystemExit("the large batch fitted")
except gpu.LambdaError as e:
    assert "memory" in str(e), e
assert live() - before < 1 * MB, (live() - before) / MB
gpu.render_batch([small])
assert live() - before < 64 * MB, (live() - before) / MB
gpu.render(fits)
""")


def test_batch_pool_is_kept_up_to_its_bound(host_hip):
    """The pool of a small batch stays (no allocation in a second call); all of a pool above 1 GiB is given
    back, counters of many iterations included."""
    host_hip(BATCH + """
before = live()
gpu.render_batch([small])
kept = live() - before
assert 0 < kept < 64 * MB
gpu.render_batch([small])
assert live() - before == kept
gpu.render_batch([fits])
assert live() - before < 1 * MB, (live() - before) / MB
gpu.render_batch([small], max_iterations=(GIB + GIB // 16) // 128)
assert live() - before < 1 * MB, (live() - before) / MB
""")


def test_counters_of_any_iteration_count_are_allocated(host_hip):
    """A job's queue counters take 128 bytes an iteration: 2^27 iterations do not fit 4 GiB and are refused
    for that (a 32-bit word count would wrap to a few bytes and the kernels would count past them)."""
    host_hip(BATCH + """
try:
    gpu.render_batch([small], max_iterations=1 << 27)
    raise SystemExit("not refused")
except gpu.LambdaError as e:
    assert "memory" in str(e), e
gpu.render_batch([small])
""")


FILM = """
def film(w, h):
    f = gpu.Film(dev, w, h)
    return f
def fails(call):
    try:
        call()
    except gpu.LambdaError as e:
        assert "memory" in str(e), e
    else:
        raise SystemExit("fitted")
"""


def test_failed_film_operations_keep_no_temporaries(host_hip):
    """Denoising, post-processing and reading an image of a film whose temporaries do not fit: what was
    obtained is given back, and the same operations on a small film go through."""
    host_hip(FILM + """
big, small = film(3600, 3000), film(64, 48)   # 165 MiB an RGBA temporary
big.read_rgba(), big.read()                   # the copier's buffers
before = live()
post, _ = abi.post_desc()
for call, temporaries in ((lambda f: f.denoise(abi.denoise_desc(), albedo=f, normal=f), 3.5), (lambda f: f.post(post), 1.5)):
    H.host_hip_budget(before + int(temporaries * 165 * MB))
    fails(lambda: call(big))
    assert live() == before, (live() - before) / MB
    call(small)
    assert live() - before < 1 * MB
    H.host_hip_budget(before + 1000 * MB)
    call(big)
    assert live() - before < 50 * MB, (live() - before) / MB  # the 8-bit image, below the bound
    before = live()
""")


def test_failed_ray_batch_keeps_no_temporaries(host_hip):
    """A ray batch whose hit records do not fit beside the rays."""
    host_hip(FILM + """
s = gpu.Scene(dev)
scene.cornell_box().push(s, abi.LIGHTS_TREE)
rays = np.zeros((5 << 20, 8), dtype=np.float32)     # 160 MiB of rays, 80 of hits
s.intersect(rays[:1000])
before = live()
H.host_hip_budget(before + 200 * MB)
fails(lambda: s.intersect(rays))
assert live() - before < 1 * MB, (live() - before) / MB
s.intersect(rays[:1000])
H.host_hip_budget(before + 400 * MB)
s.intersect(rays)
assert live() - before < 100 * MB
""")


def test_noalloc_renders_allocate_nothing_and_do_not_wait_per_bounce(host_hip):
    """lgpu_render_noalloc takes no device or pinned memory, the first call included, and its path loops read
    no counter back (their bounces publish it, as in lgpu_render): its one copy is the scene record's."""
    host_hip("""
s = gpu.Scene(dev)
scene.fog_cornell().push(s, abi.LIGHTS_TREE)
f = gpu.Film(dev, 64, 48)
before, pinned = live(), H.host_hip_pinned()
for integrator in (abi.INTEGRATOR_PATH, abi.INTEGRATOR_VOLPATH, abi.INTEGRATOR_MIS_VOLPATH):
    d = gpu.render_desc(s, f, scene.cornell_camera(64, 48), 0, 2, estimator=abi.ESTIMATOR_CORRECTED, integrator=integrator)
    copies()
    assert gpu.lib().lgpu_render_noalloc(C.byref(d), C.byref(abi.RenderStats())) == 0
    assert [c[2] for c in copies()] == [1], integrator
    assert live() == before and H.host_hip_pinned() == pinned
""")


def test_device_object_that_cannot_be_made_leaves_nothing(host_hip):
    host_hip("""
before, pinned = live(), H.host_hip_pinned()
H.host_hip_budget(before)
try:
    gpu.Device(0)
    raise SystemExit("made")
except gpu.LambdaError as e:
    assert "memory" in str(e), e
assert live() == before and H.host_hip_pinned() == pinned
H.host_hip_budget(before + MB)
d = gpu.Device(0)
d.close()
assert live() == before and H.host_hip_pinned() == pinned
""")
