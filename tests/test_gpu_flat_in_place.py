"""In-place rendering of scenes without tiles (the plain kernel and the
allocation-free call) against the oracle, bit for bit: images smaller than a wave's
8 x 8 pixels, with ragged edges and long and thin ones; one frame per launch and
several; and its counts of rays and tests against the persistent kernel's."""
import numpy as np
import pytest

from _scenes import oracle_accumulate
from ataraxia_amd import ATX_ACCEL_BVH, ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT, Renderer
from test_zz_no_alloc import DeviceArray, noalloc, reference_entry, scene

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (8, 8), (9, 7), (65, 3), (1, 130), (70, 45)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("spheres,lights,bounces,sky,kahan", [(14, 3, 6, True, False), (4, 0, 4, True, True),
                                                              (0, 2, 3, False, False), (6, 1, 0, True, False)])
def test_flat_in_place(w, h, spheres, lights, bounces, sky, kahan):
    sc = scene(200 + spheres, spheres, lights, w, h, bounces, sky=sky)
    want = oracle_accumulate(sc, 7, kahan)
    acc, img = reference_entry(sc, [3, 4], ATX_ACCEL_BVH, kahan)[-1]
    assert np.array_equal(acc.reshape(-1, 4), want[0]) and np.array_equal(img.reshape(-1), want[1].reshape(-1))
    bufs = [DeviceArray(w * h * 16), DeviceArray(w * h * 16), DeviceArray(w * h * 4)]
    try:
        for first, n in ((1, 2), (3, 5)):
            acc, img = noalloc(sc, first, n, ATX_ACCEL_BVH, kahan, bufs)
        assert np.array_equal(acc, want[0]) and np.array_equal(img, want[1].reshape(-1))
    finally:
        for b in bufs:
            b.free()


@pytest.mark.parametrize("lights", [0, 2])
def test_counts(lights):
    sc = scene(220, 9, lights, 61, 33, 5)
    print(f"case flat counts lights={lights}", flush=True)
    st = {}
    for kernel in (ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT):
        with Renderer() as r:
            r.set_kernel(kernel)
            r.on_resize(sc.camera.width, sc.camera.height)
            r.set_settings(sc.settings)
            r.set_scene(sc)
            r.render_frames(sc.camera, 1)
            st[kernel] = r.stats()
    for key in ("samples", "rays", "sphere_tests", "box_tests", "reused_rays"):
        assert st[ATX_KERNEL_PLAIN][key] == st[ATX_KERNEL_WAVEFRONT][key], key
    assert st[ATX_KERNEL_PLAIN]["sphere_tests"] == 10 * st[ATX_KERNEL_PLAIN]["rays"] > 0
