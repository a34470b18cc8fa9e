"""Sockets that are one texture lookup (no shader program), in every form they take, against the CPU oracle
path by path (1e-4 relative + 1e-6, 99.9 % of paths as in the media parity tests): textures of 1, 3 and 4
channels read as a spectrum, a broadcast channel, a real and a roughness."""
import numpy as np
import pytest

from lambda_amd import abi, gpu, scene
from tests import helpers

pytestmark = pytest.mark.gpu


def _room(channels, program):
    """The Cornell room with textured walls; program: one wall reads a shader program too."""
    rng = np.random.default_rng(channels)
    N = abi
    node, Mat = scene.node, scene.Material
    sd = scene.SceneDesc()
    shape = (7, 5) if channels == 1 else (7, 5, channels)
    t = sd.add_texture(rng.uniform(0.2, 0.8, size=shape).astype(np.float32))
    ggx = [1.0, 1.0, 1.45, *scene.COPPER_ETA, *scene.COPPER_K, 0.0]
    mats = [
        [node(N.NODE_IMAGE_COLOUR, p=[t]), node(N.NODE_LAMBERTIAN, [0])],
        [node(N.NODE_IMAGE_COLOUR, p=[t]), node(N.NODE_IMAGE_CHANNEL, p=[t, 2]), node(N.NODE_OREN_NAYAR_BRDF, [0, 1])],
        [node(N.NODE_RGB, p=(0.9, 0.9, 0.9)), node(N.NODE_IMAGE_SCALAR, p=[t]), node(N.NODE_MICROFACET_BRDF, [0, 1], p=ggx)],
        [node(N.NODE_IMAGE_CHANNEL, p=[t, 1]), node(N.NODE_LAMBERTIAN, [0])],
        [node(N.NODE_IMAGE_COLOUR, p=[t]), node(N.NODE_LAMBERTIAN, [0]), node(N.NODE_RGB, p=(0.9, 0.8, 0.7)),
         node(N.NODE_IMAGE_COLOUR, p=[t]), node(N.NODE_MICROFACET_BRDF, [2, 3], p=ggx), node(N.NODE_IMAGE_CHANNEL, p=[t, 3]),
         node(N.NODE_MIX_BSDF, [1, 4, 5])],
    ]
    if program:
        mats[3] = [node(N.NODE_CHECKER, p=[4]), node(N.NODE_SCALAR_TO_COLOUR, [0]), node(N.NODE_LAMBERTIAN, [1])]
    quads = [((-1, -1, -1), (-1, -1, 1), (1, -1, 1), (1, -1, -1)), ((-1, 1, -1), (1, 1, -1), (1, 1, 1), (-1, 1, 1)),
             ((-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1)), ((-1, -1, -1), (-1, 1, -1), (-1, 1, 1), (-1, -1, 1)),
             ((1, -1, -1), (1, -1, 1), (1, 1, 1), (1, 1, -1))]
    uv = np.array([[0.0, 0.0], [1.3, 0.1], [1.1, 1.7], [-0.4, 0.9]], dtype=np.float32)
    for q, m in zip(quads, mats):
        v, i = scene._quad(*q)
        sd.add_mesh(v, i, sd.add_material(Mat(m, bxdf=len(m) - 1)), uvs=uv)
    # an emitter that reads the texture
    v, i = scene._quad((-0.25, 0.999, -0.25), (0.25, 0.999, -0.25), (0.25, 0.999, 0.25), (-0.25, 0.999, 0.25))
    sd.add_mesh(v, i, sd.add_material(Mat([node(N.NODE_IMAGE_COLOUR, p=[t])], emission=0, intensity=12.0)), uvs=uv)
    return sd


CALLS = [(abi.INTEGRATOR_PATH, abi.SPECTRAL_HERO4, abi.ESTIMATOR_CORRECTED),
         (abi.INTEGRATOR_PATH, abi.SPECTRAL_RGB, abi.ESTIMATOR_FAITHFUL),
         (abi.INTEGRATOR_DIRECT, abi.SPECTRAL_RGB, abi.ESTIMATOR_CORRECTED),
         (abi.INTEGRATOR_VOLPATH, abi.SPECTRAL_RGB, abi.ESTIMATOR_CORRECTED),
         (abi.INTEGRATOR_MIS_VOLPATH, abi.SPECTRAL_HERO4, abi.ESTIMATOR_CORRECTED),
         (abi.INTEGRATOR_VOLPATH, abi.SPECTRAL_HERO4, abi.ESTIMATOR_FAITHFUL)]


@pytest.mark.parametrize("program", [False, True])
@pytest.mark.parametrize("channels", [1, 3, 4])
@pytest.mark.parametrize("integrator,spectral,estimator", CALLS)
def test_texture_sockets(channels, program, integrator, spectral, estimator):
    sd = _room(channels, program)
    o, _ = helpers.oracle_scene(sd)
    dev = gpu.Device(0)
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    film = gpu.Film(dev, 32, 32)
    cam = scene.cornell_camera(32, 32)
    pixels = np.tile(np.arange(1024, dtype=np.uint32), 2)
    samples = np.repeat(np.arange(2, dtype=np.uint32), 1024)
    d = gpu.render_desc(s, film, cam, 0, 2, max_bounces=6, min_bounces=3, spectral=spectral, estimator=estimator,
                        integrator=integrator)
    g = gpu.trace_paths(d, pixels, samples)
    od = helpers.desc(cam, 0, 2, 6, 3, spectral, estimator)
    od.integrator = integrator
    c = o.trace_paths(od, 32, 32, pixels, samples)
    ok = helpers.rel_close(g[:, :4], c[:, :4], 1e-4, 1e-6).all(axis=1)
    assert (np.abs(c[:, :3]).sum(axis=1) > 0).mean() > 0.3
    assert ok.mean() >= 0.999
    del keep
