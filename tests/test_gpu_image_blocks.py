"""The page-locked buffers that a renderer lends to its images: an image
keeps its pixels whatever is rendered or closed after it, and buffers come
back once an image and its views are gone."""
import gc
import threading

import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes

pytestmark = pytest.mark.gpu


def renderer(res=48, seed=3):
    return px.SamplerRenderer(scenes.direct_lighting_scene(level=2), scenes.pinhole(res, res),
                              px.StratifiedSampler(1, 1, seed), px.DirectLightingIntegrator(1))


@pytest.mark.parametrize("res", [48, 640])
def test_images_outlive_frames_and_renderers(res):
    r = renderer(res)
    first = r.render()[0]
    want = first.copy()
    kept = [r.render("plain" if k % 2 else "batched")[0] for k in range(5)]  # more than the buffers
    for img in kept:
        assert img.dtype == np.float32 and img.flags.c_contiguous and img.flags.writeable and img.shape == (res, res, 3)
        assert np.array_equal(img, want)
    assert len({img.__array_interface__["data"][0] for img in kept + [first]}) == 6
    kept[0][:] = -1.0  # the caller's to write
    view = kept[1][10:20]
    del kept[1], img
    gc.collect()
    again = r.render()[0]
    assert np.array_equal(again, want) and np.array_equal(view, want[10:20])
    r.close()
    gc.collect()
    assert np.array_equal(again, want) and np.array_equal(view, want[10:20]) and (kept[0] == -1.0).all()
    del again, view, kept
    gc.collect()


def test_buffers_are_bounded_and_come_back():
    r = renderer()
    r.render()
    blocks = r._images
    for _ in range(20):
        img = r.render()[0]
    assert len(blocks.free) == 1 and sum(b is not None for b in blocks.free) <= 1
    imgs = [r.render()[0] for _ in range(4)]
    assert len(blocks.free) == 0
    del img, imgs
    gc.collect()
    assert len(blocks.free) == 2
    r.close()
    assert len(blocks.free) == 0


def test_renderers_of_several_threads():
    want = renderer().render()[0].copy()
    bad = []

    def work():
        r = renderer()
        for _ in range(10):
            if not np.array_equal(r.render()[0], want):
                bad.append(1)
        r.close()

    ts = [threading.Thread(target=work) for _ in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
