"""The per-ray traversal kernel puts a reached leaf aside and walks on until a
second one: against the oracle at every refill threshold (0: only when all
lanes are done), stack depth and kind of tree, and at hits of t = NaN, after
which it starts again and tests nothing early."""
import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from gpu_util import F32, FMAX, check_any, check_closest, mesh_pair, random_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 1, 50, 100])
def per_ray(request):
    px.set_tuning("batched", "closest", 256, 0, request.param, "ray", stack=8)
    px.set_tuning("batched", "any", 128, 1, request.param, "ray", stack=8, lanes=1)
    yield
    px.reset_tuning()


@pytest.mark.parametrize("n,max_prims,split", [(1, 1, "sah"), (2, 1, "sah"), (5, 8, "sah"), (3000, 1, "middle"),
                                               (3000, 7, "equal"), (40000, 2, "sah")])
def test_trees_of_one_leaf_to_many(per_ray, n, max_prims, split):
    v, idx = scenes.random_triangles(n, 13, 0.05, 0.4)
    bvh, orc = mesh_pair(v, idx, split, max_prims)
    for rays in (1, 63, 30000):
        o, d = random_rays(rays, 5 + rays)
        check_closest(bvh, orc, o, d)
        check_closest(bvh, orc, o, d, mint=0.3, maxt=1.1)
        check_any(bvh, orc, o, d)
        check_any(bvh, orc, o, d, mint=0.3, maxt=1.1)
    px.synchronize()


def test_hits_at_nan_distance(per_ray):
    # triangles of size 1e-20 with a corner at the rays' origin: 1/div is
    # infinite and t = 0 * inf = NaN, after which nothing limits tmax
    v, idx = scenes.random_triangles(400, 5, 0.1, 0.6)
    e = 1e-20
    tiny = np.array([[e, 0, 0], [0, e, 0], [0, 0, 0], [0, e, 0], [0, 0, e], [0, 0, 0]], F32)
    idx = np.concatenate([idx, np.arange(6, dtype=np.uint32).reshape(2, 3) + len(v)])
    bvh, orc = mesh_pair(np.concatenate([v, tiny]), idx, "sah")
    _, d = random_rays(3000, 6)
    o = np.zeros_like(d)
    for maxt in (FMAX, 1.0):
        ref = orc.intersect(o, d, 0.0, maxt, nthreads=4)
        hits = bvh.intersect(px.RayBatch(o, d, 0.0, maxt), "batched")
        assert np.array_equal(hits["prim"], ref["prim"])
        nan = np.isnan(ref["t"])
        assert nan.any() and np.array_equal(np.isnan(hits["t"]), nan)
        hit = (ref["prim"] != px.NO_HIT) & ~nan
        assert np.array_equal(hits["t"][hit].view(np.uint32), ref["t"][hit].view(np.uint32))
    px.synchronize()


@pytest.mark.parametrize("block,bpc", [(64, 1), (256, 1), (128, 3)])
def test_claims_at_the_edges_of_a_launch(block, bpc):
    # every ray taken once: counts around the waves' first chunks, the first
    # claims of each counter and the change of the chunk size
    v, idx = scenes.random_triangles(3000, 13, 0.05, 0.4)
    bvh, orc = mesh_pair(v, idx, "sah", 1)
    lanes = 256 * bpc * block  # of the launch: 256 CUs
    px.set_tuning("batched", "closest", block, bpc, 60, "ray")
    px.set_tuning("batched", "any", block, bpc, 60, "ray", lanes=1)
    try:
        for n in (63, 65, lanes - 1, lanes, lanes + 1, lanes + 64 * 7 + 1, lanes + 64 * 9, 3 * lanes - 5,
                  32 * lanes - 1, 32 * lanes + 129):
            if n > 1 << 20:
                continue
            o, d = random_rays(n, n)
            check_closest(bvh, orc, o, d)
            check_any(bvh, orc, o, d)
    finally:
        px.reset_tuning()
    px.synchronize()
