"""The volumetric stage's rays in kernels of their own, one scene for each way a ray can be resolved,
against the CPU oracle path by path (1e-4 relative + 1e-6, 99.9 % of paths as in the media parity tests)."""
import math

import numpy as np
import pytest

from lambda_amd import abi, gpu, scene
from tests import helpers

pytestmark = pytest.mark.gpu


def _sky_and_grid():
    """Emissive quads, textured surfaces, a cloud crossed by most rays, and a sky (rays that escape)."""
    sd, _ = scene.inverse_scene(tex_res=16, grid_res=8, n_spheres=2, ground_res=6, n_light_quads=8)
    return sd, scene.inverse_camera(40, 40)


def _spots():
    """Point and spot lights only: nothing a sampled direction can reach."""
    sd = scene.media_scene(res=8, n_points=3)
    v, i = scene._quad((-3, -1.2, 3), (3, -1.2, 3), (3, -1.2, -3), (-3, -1.2, -3))
    sd.add_mesh(v, i, sd.add_material(scene.lambertian((0.6, 0.5, 0.4))))
    sd.add_spot_light((1.0, 2.5, 0.0), (-0.3, -1.0, 0.0), math.radians(40.0), math.radians(10.0), 20.0)
    return sd, scene.media_camera(40, 40)


SCENES = {
    "no_media": lambda: (scene.cornell_box(), scene.cornell_camera(40, 40)),
    "sky_and_grid": _sky_and_grid,
    "spots": _spots,
    "programs": lambda: (scene.procedural_cornell(), scene.cornell_camera(40, 40)),
}


@pytest.mark.parametrize("integrator", [abi.INTEGRATOR_VOLPATH, abi.INTEGRATOR_MIS_VOLPATH])
@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("lights", [abi.LIGHTS_TREE, abi.LIGHTS_POWER])
def test_ray_kinds(name, integrator, lights):
    sd, cam = SCENES[name]()
    o, _ = helpers.oracle_scene(sd, lights)
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = sd.push(s, lights)
    film = gpu.Film(dev, 40, 40)
    pixels = np.tile(np.arange(1600, dtype=np.uint32), 2)
    samples = np.repeat(np.arange(2, dtype=np.uint32), 1600)
    d = gpu.render_desc(s, film, cam, 0, 2, max_bounces=8, min_bounces=3, estimator=abi.ESTIMATOR_CORRECTED,
                        integrator=integrator)
    g = gpu.trace_paths(d, pixels, samples)
    od = helpers.desc(cam, 0, 2)
    od.integrator = integrator
    c = o.trace_paths(od, 40, 40, pixels, samples)
    ok = helpers.rel_close(g[:, :3], c[:, :3], 1e-4, 1e-6).all(axis=1)
    assert (np.abs(c[:, :3]).sum(axis=1) > 0).mean() > 0.05
    assert ok.mean() >= 0.999
    del keep
