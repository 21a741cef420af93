"""Queries with several lanes per ray, batched launches of up to 2^20 rays.
Closest hit (k_closest_group) against the oracle, bit for bit, at the sizes,
trees and rays where its ordered commit could go wrong, and a host model of
its stack; occlusion's bit words (k_occlude_group), which its blocks write whole."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import pbrt_rust_amd as px
import test_group_stack_model as model
from pbrt_rust_amd import scenes
from gpu_util import F32, check_closest, mesh_pair, random_rays

GSTK_CL = {4: 96, 8: 96, 16: 160, 32: 192}  # stack entries of a closest-hit group, by its lanes


@pytest.fixture(params=[0, 1, 4, 8, 16])
def lanes(request):
    # 0: the rule by launch size; 1: the per-ray kernel
    px.lib().pbrtx_set_ray_lanes(request.param)
    yield request.param
    px.reset_tuning()


def tied_rays(v, idx, n, seed):
    """Rays at an icosphere's vertices and edge midpoints: several faces share the closest t."""
    rng = np.random.default_rng(seed)
    f = idx[rng.integers(0, len(idx), n)]
    tgt = np.where((rng.random(n) < 0.5)[:, None], v[f[:, 0]], 0.5 * (v[f[:, 0]] + v[f[:, 1]]))
    o = (rng.normal(size=(n, 3)) * 1.2).astype(F32)
    return o, (tgt - o).astype(F32)


@pytest.mark.gpu
@pytest.mark.parametrize("max_prims,split", [(1, "sah"), (4, "middle"), (8, "equal")])
def test_ties_and_leaves_of_several_prims(lanes, max_prims, split):
    v, idx = scenes.icosphere(4)
    v, idx = v.astype(F32), idx.astype(np.uint32)
    bvh, orc = mesh_pair(v, idx, split, max_prims)
    o, d = tied_rays(v, idx, 20000, 3)
    check_closest(bvh, orc, o, d)
    check_closest(bvh, orc, o, d, mint=1e-3, maxt=0.9999)
    # duplicated faces: every hit is tied
    idx2 = np.concatenate([idx, idx[::-1]])
    bvh, orc = mesh_pair(v, idx2, split, max_prims)
    check_closest(bvh, orc, o, d)
    px.synchronize()


@pytest.mark.gpu
def test_ragged_counts(lanes):
    v, idx = scenes.random_triangles(5000, 21, 0.05, 0.3)
    bvh, orc = mesh_pair(v, idx, "sah", 2)
    for n in (1, 3, 4, 7, 8, 9, 15, 17, 31, 63, 65, 255, 257, 4096, 4097, 24577):
        o, d = random_rays(n, 100 + n)
        check_closest(bvh, orc, o, d)
    px.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("n,split", [(100, "middle"), (50, "middle"), (2000, "sah")])
def test_deep_and_wide_frontiers(lanes, n, split):
    # a chain too deep for the group stack (61 levels: the per-ray kernel), one
    # that just fits, and thin triangles whose boxes all overlap (the stack
    # fills to its bound and continues depth first)
    if split == "middle":
        xs = 2.0 ** np.arange(n)
        v = np.concatenate([np.array([[x, 0, 0], [x, 1, 0], [x, 0, 1]]) for x in xs]).astype(F32)
        o = np.concatenate([np.full((3000, 1), -1.0), np.random.default_rng(n).uniform(0.05, 0.7, (3000, 2))], 1)
        d = np.tile(np.array([[1, 0, 0]], F32), (3000, 1))
    else:
        rng = np.random.default_rng(9)
        z = np.sort(rng.uniform(-1, 1, n))
        v = np.concatenate([np.array([[-1, -1, q], [1, 1, q], [-0.95, -1, q]]) for q in z]).astype(F32)
        o = np.concatenate([rng.uniform(-1, 1, (4000, 2)), np.full((4000, 1), -2.0)], 1)
        o[::3, 0] = rng.uniform(-0.99, -0.97, len(o[::3]))
        o[::3, 1] = o[::3, 0] - 0.005
        d = np.concatenate([rng.normal(0, 1e-3, (4000, 2)), np.ones((4000, 1))], 1)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    bvh, orc = mesh_pair(v, idx, split)
    check_closest(bvh, orc, o.astype(F32), d.astype(F32))
    px.synchronize()  # raises if a traversal stack overflowed


@pytest.mark.gpu
def test_hits_at_nan_distance(lanes):
    # triangles of size 1e-20 with a corner at the rays' origin: 1/div is
    # infinite and t = 0 * inf = NaN, after which nothing limits tmax; the
    # last prim that the reference meets wins
    if lanes == 1:
        pytest.skip("the per-ray kernel leaves out slots by the tmax of the time their record was read")
    v, idx = scenes.random_triangles(400, 5, 0.1, 0.6)
    e = 1e-20
    tiny = np.array([[e, 0, 0], [0, e, 0], [0, 0, 0], [0, e, 0], [0, 0, e], [0, 0, 0]], F32)
    idx = np.concatenate([idx, np.arange(6, dtype=np.uint32).reshape(2, 3) + len(v)])
    v = np.concatenate([v, tiny])
    bvh, orc = mesh_pair(v, idx, "sah")
    _, d = random_rays(3000, 6)
    o = np.zeros_like(d)
    ref = orc.intersect(o, d, 0.0, float(np.finfo(np.float32).max), nthreads=4)
    for path in ("plain", "batched"):
        hits = bvh.intersect(px.RayBatch(o, d), path)
        assert np.array_equal(hits["prim"], ref["prim"]), path
        fin = np.isfinite(ref["t"]) & (ref["prim"] != px.NO_HIT)
        assert np.array_equal(hits["t"][fin].view(np.uint32), ref["t"][fin].view(np.uint32))
        assert np.isnan(hits["t"][np.isnan(ref["t"])]).all()
    assert np.isnan(ref["t"]).any() and fin.any()
    px.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("g", [0, 1, 4, 8, 16])
def test_occlusion_words_are_written_whole(block, g):
    # occlusion bits into words that hold ones before the call: every word of
    # the rays is written, the bits past the last ray are zero, and the word
    # after them is left alone
    v, idx = scenes.random_triangles(4000, 31, 0.05, 0.2)
    bvh, orc = mesh_pair(v, idx)
    try:
        px.set_tuning("batched", "any", block, 0, 60, "ray", lanes=g)
        for n in (1, 7, 8, 9, 16, 31, 32, 33, 63, 64, 65, 129, 1000, 4096, 4097, 16385, 33001):
            o, d = random_rays(n, 200 + n)
            rays = px.DeviceBuffer.from_array(px.RayBatch(o, d, 0.0, 0.7).a)
            nw = (n + 31) // 32
            bits = px.DeviceBuffer.from_array(np.full(nw + 1, 0xFFFFFFFF, np.uint32))
            bvh.intersect_p_device(rays.ptr, n, bits.ptr)
            px.synchronize()
            got = bits.download(np.uint32, nw + 1)
            assert got[nw] == 0xFFFFFFFF
            got = np.unpackbits(got[:nw].view(np.uint8), bitorder="little")
            ref, _ = orc.intersect_p(o, d, 0.0, 0.7, nthreads=4)
            assert np.array_equal(got[:n], ref.astype(np.uint8)) and not got[n:].any(), n
    finally:
        px.reset_tuning()


def query_all(bvh, rec, path):
    n = len(rec)
    rays, hits = px.DeviceBuffer.from_array(rec), px.DeviceBuffer(16 * n)
    bits = px.DeviceBuffer(4 * ((n + 31) // 32))
    bvh.intersect_p_device(rays.ptr, n, bits.ptr, path)
    bvh.intersect_device(rays.ptr, n, hits.ptr, path)
    px.synchronize()  # raises if a traversal stack overflowed
    return hits.download(np.uint32, 4 * n), rays.download(np.uint32, 8 * n), bits.download(np.uint32, (n + 31) // 32)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(1 << 20) + 1, 1500000])
@pytest.mark.parametrize("scene", ["soup", "ties", "overlap"])
def test_launches_that_hand_their_last_rays_over(scene, n):
    # past 2^20 rays one lane takes a ray and each wave hands its last rays to
    # the several-lane kernels: the same bits as the plain path, in a soup, at
    # tied hits, and among boxes that all overlap (stacks too long for a record)
    rng = np.random.default_rng(77)
    if scene == "ties":
        v, idx = scenes.icosphere(5)
        v, idx = v.astype(F32), idx.astype(np.uint32)
        o, d = tied_rays(v, idx, n, 78)
    elif scene == "soup":
        v, idx = scenes.random_triangles(30000, 79)
        o, d = random_rays(n, 80)
    else:
        k = 5000
        z = np.sort(rng.uniform(-1, 1, k))
        v = np.stack([np.stack([np.full(k, -1), np.full(k, -1), z], 1), np.stack([np.ones(k), np.ones(k), z], 1),
                      np.stack([np.full(k, -0.95), np.full(k, -1), z], 1)], 1).reshape(-1, 3).astype(F32)
        idx = np.arange(3 * k, dtype=np.uint32).reshape(-1, 3)
        o, d = random_rays(n, 81)
        o[::4096] = (0.7, -0.7, -2.0)  # a few rays along z, through every box
        d[::4096] = (1e-4, 1e-4, 1.0)
    bvh = px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 2, "sah")
    rec = px.RayBatch(o, d, 0.0, np.where(rng.random(n) < 0.5, F32(1.1), F32(np.finfo(np.float32).max))).a
    for a, b in zip(query_all(bvh, rec, "plain"), query_all(bvh, rec, "batched")):
        assert np.array_equal(a, b)


def walk_put_back(tree, depth, G, rng):
    """model.walk with leaves that go back on the stack while a record of the same step lies before them."""
    lim = GSTK_CL[G] - 3 * depth
    assert 3 * depth + 8 <= GSTK_CL[G]
    stack, steps = [0], 0
    while stack:
        top = len(stack)
        k = min(G, top, (lim - top) // 3 if top + 6 <= lim else 1)
        taken = [stack.pop() for _ in range(k)]
        pushes, record = [], False
        for e in taken:  # in visiting order
            if e is not None:
                pushes.append(list(tree[e]))
                record = record or bool(tree[e])
            elif record and rng.random() < 0.7:
                pushes.append([None])
        for p in reversed(pushes):
            stack.extend(reversed(p))
        assert len(stack) <= GSTK_CL[G], len(stack)
        steps += 1
        assert steps < 200000
    return steps


@pytest.mark.parametrize("G", [4, 8, 16, 32])
@pytest.mark.parametrize("depth,fan", [(1, 0), (6, 4), (9, 3), (14, 2), (29, 1), (29, 2)])
def test_model_of_the_stack_bound(G, depth, fan):
    rng = random.Random(depth * 7 + fan + G)
    tree = model.chain(depth) if fan == 0 else model.bushy(depth, fan, rng, 4000)
    walk_put_back(tree, depth, G, rng)
