"""The volumetric shade stage at the edges of its 256-path blocks: a path's result does not depend on how many
paths run beside it (bit for bit, whatever the block that takes it), and the paths are the CPU oracle's
(1e-4 relative + 1e-6, 99.9 % of paths as in the media parity tests)."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene
from tests import helpers

pytestmark = pytest.mark.gpu

W = H = 32
MOST = 1500


@pytest.fixture(scope="module")
def fog():
    """(trace on the GPU, trace on the CPU) of the fog room's first `paths` paths, the first of them a bright one."""
    sd = scene.fog_cornell()
    cam = scene.cornell_camera(W, H)
    o, _ = helpers.oracle_scene(sd)
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    film = gpu.Film(dev, W, H)
    pixels = (500 + np.arange(MOST, dtype=np.uint32) * 7) % (W * H)
    samples = np.arange(MOST, dtype=np.uint32) // 3

    def on_gpu(integrator, paths):
        d = gpu.render_desc(s, film, cam, 0, 512, max_bounces=8, min_bounces=3, estimator=abi.ESTIMATOR_CORRECTED,
                            integrator=integrator)
        return gpu.trace_paths(d, pixels[:paths], samples[:paths])

    def on_cpu(integrator):
        d = helpers.desc(cam, 0, 512)
        d.integrator = integrator
        return o.trace_paths(d, W, H, pixels, samples)
    yield on_gpu, on_cpu
    del keep
    film.close()
    s.close()
    dev.close()


@pytest.mark.parametrize("integrator", [abi.INTEGRATOR_VOLPATH, abi.INTEGRATOR_MIS_VOLPATH])
@pytest.mark.parametrize("paths", [1, 63, 64, 255, 256, 257, 1000])
def test_path_counts_around_a_block(fog, integrator, paths):
    on_gpu, on_cpu = fog
    most = on_gpu(integrator, MOST)
    c = on_cpu(integrator)
    bright = np.abs(c[:, :3]).sum(axis=1) > 0
    assert bright[0] and bright[:paths].mean() > 0.3 and bright.mean() > 0.3
    assert helpers.rel_close(most[:, :3], c[:, :3], 1e-4, 1e-6).all(axis=1).mean() >= 0.999
    assert np.array_equal(on_gpu(integrator, paths), most[:paths])
