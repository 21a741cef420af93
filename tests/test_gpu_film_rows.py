"""The film's gather by rows and its bounds: images of every width about the
rows' (64 pixels less the filter's reach), reaches of 0, 1 and 2 on either
axis and past them, samples a pixel at and past the rows' limit (32), and the
samplers whose positions or counts are their own; against the oracle."""
import numpy as np
import pytest

import oracle_lib as ol
import pbrt_rust_amd as px
from pbrt_rust_amd import scenes

pytestmark = pytest.mark.gpu
GAUSS = px.Filter.gaussian


@pytest.mark.parametrize("xres,yres", [(1, 1), (3, 2), (59, 3), (60, 5), (61, 4), (64, 2), (65, 3), (121, 6)])
@pytest.mark.parametrize("xw,yw", [(2.0, 2.0), (0.4, 2.4), (1.0, 0.3), (2.5, 1.0), (3.0, 3.0)])
def test_widths_and_reaches(xres, yres, xw, yw):
    scene, cam = scenes.direct_lighting_scene(level=2), scenes.pinhole(xres, yres)
    f = GAUSS(xw, yw, 1.5)
    want = ol.render(scene, cam, dict(kind="direct", nx=2, ny=2, seed=9, light_samples=1), nthreads=4, filt=f.args())
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(2, 2, 9), px.DirectLightingIntegrator(1), filter=f)
    img, _ = r.render()
    assert np.array_equal(img.view(np.uint32), want["rgb"].view(np.uint32))
    r.close()


@pytest.mark.parametrize("sampler,nx,ny", [(0, 1, 1), (0, 7, 1), (0, 8, 4), (0, 11, 3), (1, 5, 1), (1, 32, 1), (1, 33, 1),
                                           (2, 3, 1), (2, 20, 1), (2, 40, 1)])
def test_samples_a_pixel(sampler, nx, ny):
    scene, cam = scenes.direct_lighting_scene(level=2), scenes.pinhole(70, 9)
    f = px.Filter.mitchell(2.0, 2.0, 1.0 / 3.0, 1.0 / 3.0)
    want = ol.render(scene, cam, dict(kind="direct", nx=nx, ny=ny, seed=4, light_samples=1, sampler=sampler),
                     nthreads=4, filt=f.args())
    s = (px.StratifiedSampler(nx, ny, 4), px.LDSampler(nx, 4), px.HaltonSampler(nx, 4))[sampler]
    r = px.SamplerRenderer(scene, cam, s, px.DirectLightingIntegrator(1), filter=f)
    for _ in range(2):
        img, _ = r.render()
        assert np.array_equal(img.view(np.uint32), want["rgb"].view(np.uint32))
    r.close()
