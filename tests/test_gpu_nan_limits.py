"""Hits at t = NaN under a finite maxt: nothing limits the ray from then on, so
the reference's hit may lie past maxt, in boxes that begin past it.  Every
number of lanes a ray, and rays handed over, against the reference."""
import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from gpu_util import F32, FMAX, mesh_pair, random_rays

pytestmark = pytest.mark.gpu


def nan_scene(n, lo=0.1, hi=0.6):
    """A soup and two triangles of size 1e-20 with a corner at the origin: for a
    ray from there 1/div is infinite and t = 0 * inf."""
    v, idx = scenes.random_triangles(n, 5, lo, hi)
    e = 1e-20
    tiny = np.array([[e, 0, 0], [0, e, 0], [0, 0, 0], [0, e, 0], [0, 0, e], [0, 0, 0]], F32)
    return np.concatenate([v, tiny]), np.concatenate([idx, np.arange(6, dtype=np.uint32).reshape(2, 3) + len(v)])


def same_hits(hits, rays, ref, ref_maxt, maxt):
    assert np.array_equal(hits["prim"], ref["prim"]), (maxt, int((hits["prim"] != ref["prim"]).sum()))
    nan = np.isnan(ref["t"])
    assert np.array_equal(np.isnan(hits["t"]), nan)
    hit = (ref["prim"] != px.NO_HIT) & ~nan
    assert np.array_equal(hits["t"][hit].view(np.uint32), ref["t"][hit].view(np.uint32))
    assert np.array_equal(rays.maxt[~nan].view(np.uint32), ref_maxt[~nan].view(np.uint32))
    return hit & (ref["t"] > maxt)


@pytest.mark.parametrize("maxt", [FMAX, 1.0, 0.2])
@pytest.mark.parametrize("lanes", [0, 1, 4, 8, 16, 32])
def test_limits_end_at_a_nan_hit(lanes, maxt):
    bvh, orc = mesh_pair(*nan_scene(400), "sah")
    _, d = random_rays(3000, 6)
    o = np.zeros_like(d)
    ref = orc.intersect(o, d, 0.0, maxt, nthreads=4)
    px.lib().pbrtx_set_closest_lanes(lanes)
    try:
        rays = px.RayBatch(o, d, 0.0, maxt)
        past = same_hits(bvh.intersect(rays, "batched"), rays, ref, ref["maxt"], maxt)
    finally:
        px.reset_tuning()
    assert past.any() or maxt == FMAX
    px.synchronize()


@pytest.mark.parametrize("maxt", [1.0, 0.2])
def test_limits_of_rays_handed_over(maxt):
    # past 3 * 2^17 rays and 2^13 triangles the last rays go to the several-lane kernel
    bvh, _ = mesh_pair(*nan_scene(9000, 0.02, 0.1), "sah")
    n = (1 << 20) + 777
    _, d = random_rays(n, 7)
    o = np.zeros_like(d)
    a, b = px.RayBatch(o, d, 0.0, maxt), px.RayBatch(o, d, 0.0, maxt)
    want = bvh.intersect(a, "plain")
    past = same_hits(bvh.intersect(b, "batched"), b, want, a.maxt, maxt)
    assert past.any()
    px.synchronize()
