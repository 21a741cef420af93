"""The memory of a rendered image: ordinary pages, which a forked child sees
too, filled through page-locked chunks -- images of every length around the
chunks' against the same frame copied straight into page-locked memory."""
import os
import threading

import numpy as np
import pytest

import pbrt_rust_amd as px
from pbrt_rust_amd import scenes
from pbrt_rust_amd._lib import check

pytestmark = pytest.mark.gpu

LOW, HIGH, SLOTS = 1 << 18, 1 << 20, 4  # the chunks' lengths and their number


def renderer(xres, yres=1):
    return px.SamplerRenderer(scenes.direct_lighting_scene(level=2), scenes.pinhole(xres, yres),
                              px.StratifiedSampler(1, 1, 3), px.DirectLightingIntegrator(1))


def flags(address):
    """The VmFlags of the mapping around an address."""
    inside = False
    for line in open("/proc/self/smaps"):
        word = line.split()[0]
        if not word.endswith(":"):
            lo, hi = (int(x, 16) for x in word.split("-"))
            inside = lo <= address < hi
        elif inside and word == "VmFlags:":
            return line.split()[1:]


@pytest.mark.parametrize("res", [48, 640])
def test_a_forked_child_sees_the_image(res):
    r = renderer(res, res)
    for _ in range(3):
        img = r.render()[0]
        f = flags(img.ctypes.data)
        assert f and "dc" not in f and "pf" not in f and "io" not in f, f  # dc: not inherited
    got, put = os.pipe()
    pid = os.fork()
    if pid == 0:
        try:
            os.write(put, img.tobytes()[-4000:])
        finally:
            os._exit(0)
    assert os.waitpid(pid, 0)[1] == 0
    assert os.read(got, 8000) == img.tobytes()[-4000:]
    os.close(got)
    os.close(put)
    r.close()


@pytest.mark.parametrize("pixels", [1, 2, LOW // 12, LOW // 12 + 1, LOW // 6 + 1, SLOTS * LOW // 12,
                                    SLOTS * LOW // 12 + 1, 2 * LOW, 8 * HIGH // 12 - 1, 8 * HIGH // 12 + 1, HIGH])
def test_images_around_the_chunks_lengths(pixels):
    r = renderer(pixels)
    straight = px.PinnedArray((pixels * 3,), np.float32)
    check(px.lib().pbrtx_renderer_render(r._h, 1, straight.array.ctypes.data, None))
    for _ in range(3):
        img, st = r.render()
        assert st["camera_rays"] == pixels
        assert np.array_equal(img.reshape(-1).view(np.uint32), straight.array.view(np.uint32))
    # into memory at an odd place, its neighbours left alone
    room = np.full(12 * pixels + 16, 0xA5, np.uint8)
    check(px.lib().pbrtx_renderer_render(r._h, 1, room.ctypes.data + 5, None))
    assert np.array_equal(room[5:-11].copy().view(np.uint32), straight.array.view(np.uint32))
    assert (room[:5] == 0xA5).all() and (room[-11:] == 0xA5).all()
    r.close()


def test_more_renderers_at_once_than_stages_rest():
    # each image's copy has a stage of its own, whichever renderer gives or takes it
    want = [renderer(96 + k, 640).render()[0].copy() for k in range(2)]
    bad = []

    def work(k):
        for _ in range(3):
            r = renderer(96 + k % 2, 640)
            for _ in range(4):
                if not np.array_equal(r.render()[0], want[k % 2]):
                    bad.append(k)
            r.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(12)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
