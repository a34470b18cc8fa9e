"""The film's running sums go on sample by sample, so a film is the same bits however its samples are split:
over waves of any capacity, over calls, and in a batch."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene

pytestmark = pytest.mark.gpu

W, H, SPP = 40, 30, 7

SCENES = {
    "path": (lambda: scene.cornell_box(), abi.INTEGRATOR_PATH),
    "fog": (lambda: scene.fog_cornell(), abi.INTEGRATOR_VOLPATH),
    "grid": (lambda: scene.fog_cornell("grid"), abi.INTEGRATOR_MIS_VOLPATH),
}


@pytest.mark.parametrize("spectral", [abi.SPECTRAL_RGB, abi.SPECTRAL_HERO4])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_film_does_not_depend_on_the_split(name, spectral):
    make, integrator = SCENES[name]
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = make().push(s, abi.LIGHTS_TREE)
    cam = scene.cornell_camera(W, H)

    def desc(film, a, b, capacity=0):
        return gpu.render_desc(s, film, cam, a, b, max_bounces=6, min_bounces=2, spectral=spectral, capacity=capacity,
                               estimator=abi.ESTIMATOR_CORRECTED, integrator=integrator, seed=11)

    def film(render):
        f = gpu.Film(dev, W, H)
        render(f)
        out = f.read()
        f.close()
        return out

    ref, cnt = film(lambda f: gpu.render(desc(f, 0, SPP)))
    assert (cnt == SPP).all() and (ref != 0).any()
    # waves of fewer paths than pixels, of as many, of more and no multiple, of several samples of all
    ways = [lambda f, c=c: gpu.render(desc(f, 0, SPP, c)) for c in (257, W * H - 1, W * H, W * H + 500, 3 * W * H)]
    ways.append(lambda f: [gpu.render(desc(f, a, b)) for a, b in ((0, 1), (1, 4), (4, SPP))])
    ways.append(lambda f: gpu.render_batch([desc(f, 0, SPP)], max_iterations=64))
    ways.append(lambda f: gpu.render_batch([desc(f, 0, SPP)], path_capacity=1000, branches=2, max_iterations=64))
    for k, way in enumerate(ways):
        got, n = film(way)
        assert np.array_equal(n, cnt), k
        assert np.array_equal(got, ref), (k, np.abs(got - ref).max())
    del keep
    s.close()
    dev.close()
