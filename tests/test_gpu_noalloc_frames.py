"""The allocation-free call of several frames, whose lanes keep a pixel's primary
hit from frame to frame, against the renderer's frames one launch each: bit for
bit, at frame counts on both sides of where hits are kept, with and without
tiles, lights and sky, and continuing an accumulation."""
import numpy as np
import pytest

from ataraxia_amd import ATX_ACCEL_BVH, ATX_ACCEL_NONE
from test_zz_no_alloc import DeviceArray, noalloc, reference_entry, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accel", [ATX_ACCEL_BVH, ATX_ACCEL_NONE], ids=["bvh", "every"])
@pytest.mark.parametrize("spheres,lights,bounces,sky", [(9, 2, 5, True), (9, 0, 3, False), (300, 3, 6, False),
                                                        (300, 0, 4, True), (40, 1, 1, True), (40, 33, 0, True)])
@pytest.mark.parametrize("frames", [2, 3, 17])
def test_frames_of_one_launch(frames, spheres, lights, bounces, sky, accel):
    sc = scene(70 + spheres, spheres, lights, 45, 27, bounces, sky=sky)
    n = sc.camera.width * sc.camera.height
    kahan = spheres == 300
    want = reference_entry(sc, [frames, frames], accel, kahan)
    bufs = [DeviceArray(n * 16), DeviceArray(n * 16), DeviceArray(n * 4)]
    try:
        for k in range(2):
            acc, img = noalloc(sc, 1 + k * frames, frames, accel, kahan, bufs)
            assert np.array_equal(acc.view(np.uint32), want[k][0].reshape(-1, 4).view(np.uint32))
            assert np.array_equal(img, want[k][1].reshape(-1))
    finally:
        for b in bufs:
            b.free()
