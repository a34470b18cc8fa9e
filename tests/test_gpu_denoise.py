"""Device denoiser (lgpu_film_denoise, the edge-avoiding A-Trous filter standing in for OIDN's
filter of Denoise::SetData/Process, Denoise.cpp:13-67) against the CPU checker on the same film
means, and the film write/read round trip it builds on.

Bar: |gpu - cpu| <= 1e-4 * |cpu| + 1e-6 per channel (device expf against glibc's, summed over
25 taps and several passes)."""
import numpy as np
import pytest

import oracle
from lambda_amd import abi, gpu, scene
from lambda_amd.gpu import LambdaError

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = gpu.Device(0)
    yield d
    d.close()


def _means(film):
    rgb, cnt = film.read()
    inv = np.where(cnt > 0, 1.0 / np.maximum(cnt, 1), 0.0)[..., None]
    return (rgb * inv).astype(np.float32)


def _render_films(dev, W, H):
    sd = scene.cornell_box()
    s = gpu.Scene(dev)
    keep = sd.push(s, abi.LIGHTS_TREE)
    cam = scene.cornell_camera(W, H)
    colour, normal = gpu.Film(dev, W, H), gpu.Film(dev, W, H)
    gpu.render(gpu.render_desc(s, colour, cam, 0, 4, spectral=abi.SPECTRAL_HERO4))
    gpu.render(gpu.render_desc(s, normal, cam, 0, 1, integrator=abi.INTEGRATOR_NORMAL))
    return s, keep, colour, normal


def test_film_write_read_round_trip(dev):
    W, H = 13, 9
    f = gpu.Film(dev, W, H)
    rng = np.random.default_rng(2)
    rgb = rng.random((H, W, 3))
    cnt = rng.integers(0, 5, (H, W)).astype(np.uint32)
    f.write(rgb, cnt)
    r, c = f.read()
    np.testing.assert_array_equal(r, rgb)
    np.testing.assert_array_equal(c, cnt)
    f.write(rgb)
    assert (f.read()[1] == 1).all()


@pytest.mark.parametrize("guides", ["none", "normal", "albedo+normal"])
def test_denoise_matches_oracle(dev, guides):
    W, H = 48, 40
    s, keep, colour, normal = _render_films(dev, W, H)
    albedo = None
    alb = None
    if "albedo" in guides:
        # an albedo image with texture: a checker of two reflectances
        yy, xx = np.mgrid[0:H, 0:W]
        alb = np.where(((xx // 6 + yy // 6) % 2 == 0)[..., None], [0.7, 0.6, 0.5], [0.2, 0.3, 0.25])
        albedo = gpu.Film(dev, W, H)
        albedo.write(alb)
    nrm = normal if "normal" in guides else None
    d = abi.denoise_desc(iterations=5, sigma_colour=0.8, sigma_normal=0.2, sigma_albedo=0.1, demodulate=True)
    out = gpu.Film(dev, W, H)
    colour.denoise(d, albedo=albedo, normal=nrm, out=out)
    g = _means(out)
    c = oracle.denoise(_means(colour), d, albedo=None if alb is None else alb.astype(np.float32),
                       normal=None if nrm is None else _means(normal))
    assert (out.read()[1] == 1).all()
    np.testing.assert_allclose(g, c, rtol=1e-4, atol=1e-6)
    if albedo is None:  # the filter smooths (with an albedo the checker texture is put back)
        src = _means(colour)
        assert np.abs(np.diff(g, axis=1)).mean() < 0.7 * np.abs(np.diff(src, axis=1)).mean()


def test_denoise_in_place_equals_out_of_place(dev):
    W, H = 32, 24
    s, keep, colour, normal = _render_films(dev, W, H)
    d = abi.denoise_desc(iterations=3, sigma_colour=0.5, sigma_normal=0.3)
    out = gpu.Film(dev, W, H)
    colour.denoise(d, normal=normal, out=out)
    colour.denoise(d, normal=normal)
    np.testing.assert_array_equal(colour.read()[0], out.read()[0])


def test_denoise_rejects_bad_arguments(dev):
    a, b = gpu.Film(dev, 8, 8), gpu.Film(dev, 9, 8)
    with pytest.raises(LambdaError):
        a.denoise(abi.denoise_desc(iterations=0))
    with pytest.raises(LambdaError):
        a.denoise(abi.denoise_desc(iterations=13))
    with pytest.raises(LambdaError):
        a.denoise(abi.denoise_desc(sigma_colour=-1.0))
    with pytest.raises(LambdaError):
        a.denoise(abi.denoise_desc(), normal=b)


@pytest.mark.parametrize("w,h", [(1, 1), (3, 70), (64, 16), (65, 17), (130, 33), (512, 512), (513, 512)])
@pytest.mark.parametrize("iterations", [1, 3, 6])
def test_denoise_sizes(dev, w, h, iterations):
    """Image sizes around the filter's tile (64 columns, rows a step apart) and on both sides of the size where a
    thread takes two rows, steps up to 32 rows."""
    rng = np.random.default_rng(w + h)
    films, means = [], []
    for lo, hi in ((0.0, 2.0), (0.1, 0.9), (0.0, 1.0)):
        f = gpu.Film(dev, w, h)
        f.write(rng.uniform(lo, hi, size=(h, w, 3)))
        films.append(f)
        means.append(_means(f))
    d = abi.denoise_desc(iterations=iterations, sigma_colour=0.9, sigma_normal=0.7, sigma_albedo=0.6, demodulate=True)
    out = gpu.Film(dev, w, h)
    films[0].denoise(d, albedo=films[1], normal=films[2], out=out)
    c = oracle.denoise(means[0], d, albedo=means[1], normal=means[2])
    np.testing.assert_allclose(_means(out), c, rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("w,h", [(1, 270000), (270000, 1), (1, 530000), (2, 140000)])
def test_denoise_long_images(dev, w, h):
    """Images of one or two columns or rows, with more row groups than a grid's second dimension holds blocks:
    every pixel is filtered (a constant image stays what it is)."""
    f = gpu.Film(dev, w, h)
    f.write(np.full((h, w, 3), 0.625))
    out = gpu.Film(dev, w, h)
    f.denoise(abi.denoise_desc(iterations=3, sigma_colour=0.9), out=out)
    np.testing.assert_allclose(_means(out), 0.625, rtol=1e-6)
    f.close()
    out.close()
