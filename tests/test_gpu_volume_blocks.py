"""The volumetric shade stage at the edges of its 256-path blocks, against the CPU oracle path by path
(1e-4 relative + 1e-6, 99.9 % of paths as in the media parity tests)."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", [abi.INTEGRATOR_VOLPATH, abi.INTEGRATOR_MIS_VOLPATH])
@pytest.mark.parametrize("paths", [1, 63, 64, 255, 256, 257, 1000])
def test_path_counts_around_a_block(integrator, paths):
    w, h = 32, 32
    sd = scene.fog_cornell()
    cam = scene.cornell_camera(w, h)
    o, _ = helpers.oracle_scene(sd)
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    film = gpu.Film(dev, w, h)
    pixels = np.arange(paths, dtype=np.uint32) * 7 % (w * h)
    samples = np.arange(paths, dtype=np.uint32) // 3
    d = gpu.render_desc(s, film, cam, 0, 512, max_bounces=8, min_bounces=3, estimator=abi.ESTIMATOR_CORRECTED,
                        integrator=integrator)
    g = gpu.trace_paths(d, pixels, samples)
    od = helpers.desc(cam, 0, 512)
    od.integrator = integrator
    c = o.trace_paths(od, w, h, pixels, samples)
    ok = helpers.rel_close(g[:, :3], c[:, :3], 1e-4, 1e-6).all(axis=1)
    assert (~ok).sum() <= max(1, paths // 1000)
    del keep
