"""The path tracer's per-bounce counters: paths of more bounces than the
counters have places for (32), in one chunk and in several, eager and
replayed, against the plain path and the oracle; the ray counts agree."""
import numpy as np
import pytest

import oracle_lib as ol
import pbrt_rust_amd as px
from pbrt_rust_amd import scenes

pytestmark = pytest.mark.gpu


def mirror_room():
    """A box of mirrors around the camera with a light in the ceiling: paths go on to the last bounce."""
    c = np.array([[x, y, z] for x in (-2, 2) for y in (-2, 2) for z in (-4, 4)], np.float32)
    f = np.array([[0, 1, 3], [0, 3, 2], [4, 6, 7], [4, 7, 5], [0, 4, 5], [0, 5, 1], [2, 3, 7], [2, 7, 6],
                  [0, 2, 6], [0, 6, 4], [1, 5, 7], [1, 7, 3]], np.uint32)
    lv, lf = scenes.quad([-0.5, 1.9, -0.5], [-0.5, 1.9, 0.5], [0.5, 1.9, 0.5], [0.5, 1.9, -0.5])
    v, idx = np.concatenate([c, lv]), np.concatenate([f, lf + 8])
    mat = np.zeros(len(idx), np.uint32)
    mat[4:6] = 1  # the floor is matte
    mat[12:] = 2
    light = np.full(len(idx), -1, np.int32)
    light[12:] = 0
    return dict(verts=v, idx=idx, face_mat=mat, face_light=light,
                mats=np.array([[1, 0.99, 0.99, 0.99], [0, 0.8, 0.8, 0.8], [0, 0, 0, 0]], np.float32),
                area_le=np.array([[5.0] * 3], np.float32), point_lights=np.zeros((0, 6), np.float32))


@pytest.mark.parametrize("depth", [0, 1, 31, 32, 33, 70])
def test_depths_around_the_counters_places(depth):
    scene, cam = mirror_room(), scenes.pinhole(40, 24, cam_pos=(0.3, 0.2, -1.0))
    want = ol.render(scene, cam, dict(kind="path", nx=2, ny=2, seed=5, max_depth=depth, rr_start=80), nthreads=4)
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(2, 2, 5), px.PathIntegrator(depth, 80))
    plain, sp = r.render("plain")
    assert np.array_equal(plain.view(np.uint32), want["rgb"].view(np.uint32))
    keys = ("camera_rays", "shadow_rays", "extension_rays")
    assert sp["extension_rays"] > 0 or depth == 0
    for chunk in (40 * 24 * 4, 1000):
        r.set_chunk(chunk)
        for graph in (False, True):
            r.set_graph(graph)
            for _ in range(3):
                img, st = r.render("batched")
                assert np.array_equal(img.view(np.uint32), plain.view(np.uint32))
                assert [st[k] for k in keys] == [sp[k] for k in keys]
    r.close()


def test_large_and_small_vertex_tiles_agree():
    # batches of 2^23 paths and more take vertex tiles of 2048 paths, smaller
    # ones of 512: the same radiance bit for bit
    scene, cam = mirror_room(), scenes.pinhole(512, 257, cam_pos=(0.3, 0.2, -1.0))
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(8, 8, 5), px.PathIntegrator(3, 3))
    out = []
    for chunk in (512 * 257 * 64, (1 << 23) - 64, 1 << 20):
        r.set_chunk(chunk)
        img, st = r.render("batched")
        out.append((img.view(np.uint32).copy(), [st[k] for k in ("camera_rays", "shadow_rays", "extension_rays")]))
    assert all(np.array_equal(i, out[0][0]) and c == out[0][1] for i, c in out[1:])
    r.close()
