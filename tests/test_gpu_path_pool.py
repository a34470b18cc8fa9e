"""The path pool a device keeps between renders, over scenes whose trees need different amounts of
per-path traversal spill: a render must not depend on what was rendered before it."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene

pytestmark = pytest.mark.gpu


def _film(dev, sd, cam, w, h, spp):
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    film = gpu.Film(dev, w, h)
    gpu.render(gpu.render_desc(s, film, cam, 0, spp, max_bounces=6, min_bounces=3, estimator=abi.ESTIMATOR_CORRECTED))
    out = film.read()
    film.close()
    s.close()
    del keep
    return out


@pytest.mark.parametrize("first", [256, 512])
def test_deeper_tree_in_a_pool_sized_by_a_shallow_one(first):
    """A large render of the Cornell box sizes the pool (no spill words per path), then a smaller render of
    a deep tree grows only its spill area."""
    deep = scene.many_light_scene(n_spheres=12, ground_res=64, n_light_quads=64)
    cam = scene.many_light_camera(96, 64)
    dev = gpu.Device(0)
    ref, cnt = _film(dev, deep, cam, 96, 64, 4)
    dev.close()
    dev = gpu.Device(0)
    _film(dev, scene.cornell_box(), scene.cornell_camera(first, first), first, first, 1)
    got, got_cnt = _film(dev, deep, cam, 96, 64, 4)
    dev.close()
    assert (cnt == 4).all() and (got_cnt == 4).all()
    np.testing.assert_array_equal(got, ref)
