"""The GPU tree build at the sizes where its runs of boxes (8, 64, 512 leaves)
and its records begin and end, with equal Morton codes, and with a vertex
index out of range; checked as tests/test_gpu_lbvh.py checks it."""
import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from gpu_util import F32, random_rays
from test_gpu_lbvh import check, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 16, 17, 18, 63, 64, 65, 511, 512, 513, 520, 4095, 4097, 33000])
def test_sizes(n):
    v, idx = scenes.random_triangles(n, 300 + n, 0.1, 0.5)
    gpu, orc = pair(v, idx)
    o, d = random_rays(1500, n)
    check(gpu, orc, o, d)
    px.synchronize()


@pytest.mark.parametrize("n", [2, 9, 100, 1000])
def test_equal_codes(n):
    # triangles about a few shared centroids: runs of equal codes, split by position
    rng = np.random.default_rng(n)
    c = rng.uniform(-1, 1, (max(1, n // 50), 3))[rng.integers(0, max(1, n // 50), n)]
    u = rng.normal(0, 0.2, (n, 3))
    w = rng.normal(0, 0.2, (n, 3))
    v = np.stack([c + u, c - u, c + w], 1)
    v[:, 2] = np.clip(v[:, 2], np.minimum(v[:, 0], v[:, 1]), np.maximum(v[:, 0], v[:, 1]))  # the box's centre stays c
    gpu, orc = pair(v.reshape(-1, 3).astype(F32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))
    o, d = random_rays(1500, n)
    check(gpu, orc, o, d)
    px.synchronize()


@pytest.mark.parametrize("where", [0, 1000, 2999])
def test_index_out_of_range_is_refused(where):
    v, idx = scenes.random_triangles(1000, 5)
    idx = idx.copy()
    idx.reshape(-1)[where] = 3000
    with pytest.raises(px.PbrtxError, match="vertex index out of range"):
        px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 1, "lbvh")
    idx.reshape(-1)[where] = 0xFFFFFFFF
    with pytest.raises(px.PbrtxError, match="vertex index out of range"):
        px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 1, "lbvh")
    idx.reshape(-1)[where] = 2999
    px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 1, "lbvh").close()
