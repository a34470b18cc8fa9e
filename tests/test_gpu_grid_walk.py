"""Grid media whose walks end inside, at and past a group of voxels stepped ahead (one voxel, fewer than a
group along an axis, many), against the CPU oracle path by path (1e-4 relative + 1e-6, 99.9 % of paths as
in the media parity tests)."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene
from tests import helpers

pytestmark = pytest.mark.gpu


def _scene(shape):
    sd = scene.SceneDesc()
    dens = np.random.default_rng(5).uniform(-0.4, 1.5, size=shape).clip(0.0).astype(np.float32)
    dens.flat[0] = 1.0
    med = scene.grid_medium(sd, dens, [0.3, 0.2, 0.1], [1.5, 1.7, 1.9], 0.4, (-1.0, -1.0, -1.0), (1.0, 1.0, 1.0))
    v, i = scene.aabb((-1.0, -1.0, -1.0), (1.0, 1.0, 1.0))
    sd.add_mesh(v, i, sd.add_material(scene.passthrough(interior=med)))
    sd.add_point_light((0.0, 3.0, 0.5), 20.0)
    sd.add_point_light((0.1, 0.2, 0.0), 1.0, rgb=(1.0, 0.7, 0.4))
    return sd


@pytest.mark.parametrize("integrator", [abi.INTEGRATOR_VOLPATH, abi.INTEGRATOR_MIS_VOLPATH])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 3), (1, 7, 5), (9, 8, 17), (3, 2, 70)])
def test_grid_shapes(shape, integrator):
    w = h = 32
    sd = _scene(shape)
    o, _ = helpers.oracle_scene(sd)
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    film = gpu.Film(dev, w, h)
    cam = scene.media_camera(w, h)
    pixels = np.tile(np.arange(w * h, dtype=np.uint32), 2)
    samples = np.repeat(np.arange(2, dtype=np.uint32), w * h)
    d = gpu.render_desc(s, film, cam, 0, 2, max_bounces=8, min_bounces=3, estimator=abi.ESTIMATOR_CORRECTED,
                        integrator=integrator)
    g = gpu.trace_paths(d, pixels, samples)
    od = helpers.desc(cam, 0, 2)
    od.integrator = integrator
    c = o.trace_paths(od, w, h, pixels, samples)
    assert (np.abs(c[:, :3]).sum(axis=1) > 0).mean() > 0.05
    assert helpers.rel_close(g[:, :3], c[:, :3], 1e-4, 1e-6).all(axis=1).mean() >= 0.999
    del keep
