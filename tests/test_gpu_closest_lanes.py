"""Lanes per ray by kind of query: the occlusion setting leaves closest hit
alone, and closest hit has one of its own, under which the query suites of the
several-lane and the per-ray kernel run again."""
import numpy as np
import pytest

import pbrt_rust_amd as px
import test_gpu_group_queries as group
import test_gpu_leaf_aside as aside
import test_gpu_query as query
from pbrt_rust_amd import scenes
from pbrt_rust_amd._lib import check
from gpu_util import check_closest, mesh_pair, random_rays


def test_the_setting_takes_the_lanes_there_are():
    L = px.lib()
    for bad in (-1, 2, 3, 5, 64):
        assert L.pbrtx_set_closest_lanes(bad) < 0 and b"lanes per ray" in L.pbrtx_last_error()
    for good in (1, 4, 8, 16, 32, 0):
        assert L.pbrtx_set_closest_lanes(good) == 0


@pytest.mark.gpu
def test_occlusion_lanes_leave_closest_hit_alone():
    # 4M rays take twice as long with four lanes each as with one
    v, idx = scenes.random_triangles(200000, 1)
    bvh = px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 4, "sah")
    rays = px.DeviceBuffer.from_array(px.RayBatch(*random_rays(1 << 22, 2)).a)
    hits = px.DeviceBuffer(16 << 22)
    work = px.DeviceBuffer(32 << 22)

    def ms():
        out = []
        for _ in range(7):
            check(px.lib().pbrtx_device_copy(work.ptr, rays.ptr, 32 << 22, None))
            check(px.lib().pbrtx_timer_start(None))
            bvh.intersect_device(work.ptr, 1 << 22, hits.ptr)
            t = px._lib.ctypes.c_float()
            check(px.lib().pbrtx_timer_stop(None, px._lib.ctypes.byref(t)))
            out.append(t.value)
        return sorted(out)[3]

    try:
        ms()
        alone = ms()
        px.set_tuning("batched", "any", 256, 0, 60, "ray", lanes=4)
        assert ms() < 1.3 * alone
        px.lib().pbrtx_set_closest_lanes(4)
        assert ms() > 1.3 * alone
    finally:
        px.reset_tuning()


@pytest.fixture(params=[1, 4, 8, 16, 32])
def lanes(request):
    px.lib().pbrtx_set_closest_lanes(request.param)
    yield request.param
    px.reset_tuning()


@pytest.mark.gpu
@pytest.mark.parametrize("max_prims,split", [(1, "sah"), (4, "middle"), (8, "equal")])
def test_ties_and_leaves(lanes, max_prims, split):
    group.test_ties_and_leaves_of_several_prims(lanes, max_prims, split)
    v, idx = scenes.random_triangles(20000, 40 + max_prims)
    bvh, orc = mesh_pair(v, idx, split, max_prims)
    o, d = random_rays(30000, 41)
    check_closest(bvh, orc, o, d)
    px.synchronize()


@pytest.mark.gpu
def test_counts_and_frontiers(lanes):
    group.test_ragged_counts(lanes)
    for n, split in ((100, "middle"), (50, "middle"), (2000, "sah")):
        group.test_deep_and_wide_frontiers(lanes, n, split)


@pytest.mark.gpu
def test_query_suite(lanes):
    query.test_random_scene_parity("batched", "sah")
    query.test_edge_cases("batched")
    query.test_grazing_rays_on_box_planes("batched")
    query.test_mixed_finite_and_infinite_inverse_directions("batched")
    query.test_deep_tree_uses_spill_stack("batched")
    query.test_mixed_triangles_and_spheres("batched")
    query.test_eight_spheres_prim_ids("batched", "equal")
    query.test_paths_agree_at_full_size()
    px.synchronize()


@pytest.fixture
def one_lane():
    # (kept by set_tuning until reset_tuning)
    px.lib().pbrtx_set_closest_lanes(1)
    px.lib().pbrtx_set_ray_lanes(1)
    yield
    px.reset_tuning()


@pytest.mark.gpu
@pytest.mark.parametrize("stack", [8, 24])
def test_stack_depths_of_the_per_ray_kernel(one_lane, stack):
    query.test_stack_depths_match_oracle(stack)


@pytest.mark.gpu
@pytest.mark.parametrize("refill", [0, 1, 50, 100])
def test_leaves_put_aside_at_one_lane(one_lane, refill):
    px.set_tuning("batched", "closest", 256, 0, refill, "ray", stack=8)
    px.set_tuning("batched", "any", 128, 1, refill, "ray", stack=8)
    for n, max_prims, split in ((1, 1, "sah"), (2, 1, "sah"), (5, 8, "sah"), (3000, 1, "middle"), (3000, 7, "equal"),
                                (40000, 2, "sah")):
        aside.test_trees_of_one_leaf_to_many(None, n, max_prims, split)
    aside.test_hits_at_nan_distance(None)


@pytest.mark.gpu
@pytest.mark.parametrize("block,bpc", [(64, 1), (256, 1), (128, 3)])
def test_claims_at_one_lane(one_lane, block, bpc):
    aside.test_claims_at_the_edges_of_a_launch(block, bpc)
