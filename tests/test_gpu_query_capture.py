"""Queries captured in a HIP graph.  A stream's scratch depends on the scene
alone: after any call of that size of tree a larger one can be captured, and a
captured one stays good whatever is called on its stream afterwards."""
import ctypes

import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from pbrt_rust_amd._lib import check
from gpu_util import F32, random_rays

pytestmark = pytest.mark.gpu

N = (1 << 20) + 4321


class Stream:
    """A stream to capture (the HIP runtime that the library is linked to)."""

    def __init__(self):
        self.hip = px.lib()
        self.s = ctypes.c_void_p()
        self.ok(self.hip.hipStreamCreate(ctypes.byref(self.s)))

    @staticmethod
    def ok(e):
        assert e == 0, "HIP error %d" % e

    def capture(self, body):
        g, x = ctypes.c_void_p(), ctypes.c_void_p()
        self.ok(self.hip.hipStreamBeginCapture(self.s, 0))
        try:
            body()
        finally:
            e = self.hip.hipStreamEndCapture(self.s, ctypes.byref(g))
        self.ok(e)
        self.ok(self.hip.hipGraphInstantiate(ctypes.byref(x), g, None, None, ctypes.c_size_t(0)))
        return x

    def replay(self, x):
        self.ok(self.hip.hipGraphLaunch(x, self.s))
        self.sync()

    def sync(self):
        self.ok(self.hip.hipStreamSynchronize(self.s))


class Query:
    def __init__(self, bvh, o, d, kind):
        self.bvh, self.n, self.kind = bvh, len(o), kind
        self.rec = px.RayBatch(o, d, 0.0, F32(0.9) if kind == "any" else F32(np.finfo(F32).max)).a
        self.rays = px.DeviceBuffer.from_array(self.rec)
        self.words = 4 * self.n if kind == "closest" else (self.n + 31) // 32
        self.out = px.DeviceBuffer(4 * self.words)

    def run(self, path="batched", stream=None):
        f = self.bvh.intersect_device if self.kind == "closest" else self.bvh.intersect_p_device
        f(self.rays.ptr, self.n, self.out.ptr, path, stream)

    def fresh(self):
        self.rays.upload(self.rec)
        self.out.upload(np.full(self.words, 0xA5A5A5A5, np.uint32))

    def result(self):
        return self.out.download(np.uint32, self.words).copy()

    def plain(self):
        self.fresh()
        self.run("plain")
        px.synchronize()
        return self.result()


def same_on_replays(st, graph, q, want, between=lambda: None):
    for _ in range(3):
        q.fresh()
        st.replay(graph)
        assert np.array_equal(q.result(), want)
        between()


@pytest.mark.parametrize("kind", ["closest", "any"])
@pytest.mark.parametrize("warm", [1000, N])
def test_a_large_call_captured_after_a_small_one(kind, warm):
    v, idx = scenes.random_triangles(40000, 3)
    bvh = px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 2, "sah")
    st = Stream()
    w = Query(bvh, *random_rays(warm, 4), kind)
    w.run(stream=st.s)
    st.sync()
    q = Query(bvh, *random_rays(N, 5), kind)
    want = q.plain()
    x = st.capture(lambda: q.run(stream=st.s))
    same_on_replays(st, x, q, want, between=lambda: (w.run(stream=st.s), st.sync()))
    # eager on the stream afterwards, and the graph again
    q.fresh()
    q.run(stream=st.s)
    st.sync()
    assert np.array_equal(q.result(), want)
    same_on_replays(st, x, q, want)
    px.synchronize()


def test_captured_spills_outlive_larger_calls():
    # a chain whose stacks spill, one lane a ray, captured; then a call past
    # 2^20 rays on the same stream, whose rays are handed over
    n = 60
    xs = 2.0 ** np.arange(n)
    v = np.concatenate([np.array([[x, 0, 0], [x, 1, 0], [x, 0, 1]]) for x in xs]).astype(F32)
    sv, _ = scenes.random_triangles(9000, 8)
    v = np.concatenate([v, sv]).astype(F32)
    idx = np.arange(len(v), dtype=np.uint32).reshape(-1, 3)
    bvh = px.BVHAccelerator([px.Primitive.simple(px.TriangleMesh(None, None, False, idx, v))], 1, "middle")
    o = np.concatenate([np.full((3000, 1), -1.5), np.random.default_rng(1).uniform(0.05, 0.7, (3000, 2))], 1).astype(F32)
    d = np.tile(np.array([[1, 0, 0]], F32), (3000, 1))
    st = Stream()
    px.set_tuning("batched", "closest", 256, 0, 60, "ray", stack=8)
    px.lib().pbrtx_set_closest_lanes(1)
    try:
        q = Query(bvh, o, d, "closest")
        want = q.plain()
        q.run(stream=st.s)
        st.sync()
        x = st.capture(lambda: q.run(stream=st.s))
    finally:
        px.reset_tuning()
    px.set_tuning("batched", "closest", 256, 0, 60, "ray", stack=8)
    try:
        big = Query(bvh, *random_rays(N, 6), "closest")
        big_want = big.plain()

        def call():
            big.fresh()
            big.run(stream=st.s)
            st.sync()
            assert np.array_equal(big.result(), big_want)
        same_on_replays(st, x, q, want, between=call)
    finally:
        px.reset_tuning()
    px.synchronize()
