"""Camera-ray packets: frames whose samples, strata and widths are and are not
powers of two, and hit lists that fill a wave's buffer exactly or end short,
against the oracle bit for bit; rays the sign-ordered box test must refuse
(every 1/d zero or NaN) in the packet scheme; and, on the host, the division
by the image width as one product."""
import numpy as np
import pytest

import oracle_lib as ol
import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from gpu_util import F32, FMAX, mesh_pair, random_rays


@pytest.mark.parametrize("xres", [1, 2, 3, 7, 480, 1000, 1920, 4095, 65521, 1 << 20, (1 << 24) - 1])
def test_pixel_split_is_exact(xres):
    rng = np.random.default_rng(xres)
    q = rng.integers(0, (1 << 32) // xres, 4000, dtype=np.uint64)
    pix = np.concatenate([q * xres, q * xres + (xres - 1), rng.integers(0, 1 << 32, 4000, dtype=np.uint64)])
    pix = pix[pix < (1 << 32)]
    y = ((pix.astype(np.float64) + 0.5) * (1.0 / np.float64(xres))).astype(np.uint64)
    assert np.array_equal(y, pix // np.uint64(xres))


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,nx,ny", [(1, 1, 1, 1), (33, 7, 1, 1), (64, 8, 1, 1), (20, 12, 3, 1), (20, 12, 2, 3),
                                       (24, 10, 4, 1), (24, 10, 1, 4), (16, 9, 8, 8), (9, 16, 16, 4)])
@pytest.mark.parametrize("kind", ["direct", "path"])
def test_frames_match_the_oracle(w, h, nx, ny, kind):
    scene, cam = scenes.direct_lighting_scene(level=2), scenes.pinhole(w, h)
    integ = dict(kind=kind, nx=nx, ny=ny, seed=11, light_samples=2, max_depth=2, rr_start=3)
    want = ol.render(scene, cam, integ, nthreads=4)["rgb"].view(np.uint32)
    it = px.DirectLightingIntegrator(2) if kind == "direct" else px.PathIntegrator(2, 3)
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(nx, ny, 11), it)
    for chunk in (None, 100 * nx * ny, 1000):
        if chunk:
            r.set_chunk(chunk)
        img, _ = r.render("batched")
        assert np.array_equal(img.view(np.uint32), want)
    r.close()


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(64, 8), (64, 12), (64, 16), (64, 520), (61, 523)])
def test_hit_lists_of_whole_and_partial_buffers(w, h):
    # a wall across the whole view: every packet hits with all its lanes
    v = np.array([[-50, -50, 3], [50, -50, 3], [50, 50, 3], [-50, 50, 3]], F32)
    lv, lf = scenes.quad([-0.5, 1.9, -0.5], [-0.5, 1.9, 0.5], [0.5, 1.9, 0.5], [0.5, 1.9, -0.5])
    idx = np.concatenate([np.array([[0, 2, 1], [0, 3, 2]], np.uint32), lf + 4])
    scene = dict(verts=np.concatenate([v, lv]), idx=idx, face_mat=np.array([0, 0, 1, 1], np.uint32),
                 face_light=np.array([-1, -1, 0, 0], np.int32),
                 mats=np.array([[0, 0.7, 0.7, 0.7], [0, 0, 0, 0]], F32), area_le=np.array([[5.0] * 3], F32),
                 point_lights=np.zeros((0, 6), F32))
    cam = scenes.pinhole(w, h, cam_pos=(0.0, 0.0, -1.0))
    want = ol.render(scene, cam, dict(kind="path", nx=4, ny=4, seed=3, max_depth=1, rr_start=3), nthreads=8)
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(4, 4, 3), px.PathIntegrator(1, 3))
    for _ in range(2):
        img, _ = r.render("batched")
        assert np.array_equal(img.view(np.uint32), want["rgb"].view(np.uint32))
    r.close()


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["all_inf", "inf_and_nan", "zeros", "mixed"])
def test_packets_with_rays_without_a_finite_slope(case):
    rng = np.random.default_rng(4)
    v = rng.uniform(-1, 1, (300, 3)).astype(F32)
    bvh, orc = mesh_pair(v, rng.integers(0, 300, (200, 3)).astype(np.uint32))
    o, d = random_rays(257, 9)
    k = np.arange(257) % 3 == 0 if case == "mixed" else np.ones(257, bool)
    if case == "all_inf":
        d[k] = np.inf
    elif case == "inf_and_nan":
        d[k] = (np.inf, np.nan, -np.inf)
    elif case == "zeros":
        d[k] = (0.0, -0.0, 1.0)
    else:
        d[k] = (np.nan, np.nan, np.nan)
    px.set_tuning("batched", "closest", 256, 0, 0, "packet")
    try:
        rays = px.RayBatch(o, d)
        hits = bvh.intersect(rays, "batched")
    finally:
        px.reset_tuning()
    ref = orc.intersect(o, d, 0.0, FMAX, nthreads=4)
    assert np.array_equal(hits["prim"], ref["prim"])
    h = ref["prim"] != px.NO_HIT
    for f in ("t", "b1", "b2"):  # a NaN's sign and payload are not the IEEE operations' to fix
        a, b = hits[f][h], ref[f][h]
        nan = np.isnan(b)
        assert np.array_equal(np.isnan(a), nan) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))
