"""Captured frames of one path outlive the other path's: on a tree whose
stacks spill, the batched path needs more spill than the plain one, and the
renderer's stream gets it anew."""
import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes

pytestmark = pytest.mark.gpu


def test_frames_of_both_paths_on_a_deep_tree():
    n = 60
    xs = 2.0 ** np.arange(n)
    v = np.concatenate([np.array([[x, 0, 0], [x, 1, 0], [x, 0, 1]]) for x in xs]).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    scene = dict(verts=v, idx=idx, face_mat=np.zeros(n, np.uint32), face_light=np.full(n, -1, np.int32),
                 mats=np.array([[0, 0.5, 0.6, 0.7]], np.float32), area_le=np.zeros((0, 3), np.float32),
                 point_lights=np.array([[-2.0, 0.4, 0.4, 9, 9, 9]], np.float32))
    cam = scenes.look_at(64, 48, (-3.0, 0.4, 0.3), (1.0, 0.3, 0.3))
    r = px.SamplerRenderer(scene, cam, px.StratifiedSampler(2, 2, 3), px.PathIntegrator(3, 3), split="middle")
    want = r.render("plain")[0].copy()
    assert want.any()
    r.set_graph(True)
    for path in ("plain", "plain", "plain", "batched", "plain", "batched", "batched", "plain", "plain", "batched"):
        assert np.array_equal(r.render(path)[0].view(np.uint32), want.view(np.uint32)), path
    r.close()
