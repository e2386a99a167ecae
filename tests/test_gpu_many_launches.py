"""Calls of more launches than a call keeps queues (1024) or table entries (64,
allocation-free call): with accumulation off every frame is a launch that
starts over at frame 1, so the results are those of one frame."""
import numpy as np
import pytest

from ataraxia_amd import ATX_ACCEL_BVH, ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT, Renderer, Settings
from test_zz_no_alloc import DeviceArray, noalloc, scene

pytestmark = pytest.mark.gpu


def flickering(spheres):
    sc = scene(51, spheres, 2, 24, 16, 4, sky=True)
    sc.settings = Settings(False, True, 4)
    return sc


def render(sc, kernel, frames):
    print(f"case launches kernel={kernel} spheres={len(sc.spheres)} frames={frames}", flush=True)
    with Renderer() as r:
        r.set_kernel(kernel)
        r.on_resize(sc.camera.width, sc.camera.height)
        r.set_settings(sc.settings)
        r.set_scene(sc)
        r.render_frames(sc.camera, frames)
        return r.get_accumulation().reshape(-1, 4), r.get_image().reshape(-1), r.stats()


@pytest.mark.parametrize("kernel", [ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT], ids=["plain", "wavefront"])
@pytest.mark.parametrize("frames", [1024, 1025])
def test_renderer_reuses_queues(frames, kernel):
    sc = flickering(40)
    acc, img, _ = render(sc, kernel, 1)
    acc_n, img_n, st = render(sc, kernel, frames)
    assert np.array_equal(acc, acc_n) and np.array_equal(img, img_n)
    assert st["launches"] == frames and st["samples"] == frames * len(img)


@pytest.mark.parametrize("spheres", [5, 40])
@pytest.mark.parametrize("frames", [64, 65, 129])
def test_noalloc_reuses_entries(frames, spheres):
    sc = flickering(spheres)
    n = sc.camera.width * sc.camera.height
    acc, img, _ = render(sc, ATX_KERNEL_PLAIN, 1)
    bufs = [DeviceArray(n * 16), DeviceArray(n * 16), DeviceArray(n * 4)]
    try:
        acc_n, img_n = noalloc(sc, 1, frames, ATX_ACCEL_BVH, False, bufs)
        assert np.array_equal(acc, acc_n) and np.array_equal(img, img_n)
    finally:
        for b in bufs:
            b.free()
