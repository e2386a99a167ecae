"""An allocation-free call of more frames than one launch takes (4096) against the
renderer's frames one launch each, with and without tiles: bit for bit."""
import numpy as np
import pytest

from ataraxia_amd import ATX_ACCEL_BVH
from test_zz_no_alloc import DeviceArray, noalloc, reference_entry, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spheres", [5, 40])
@pytest.mark.parametrize("frames", [4096, 4097, 8199])
def test_frames_past_one_launch(frames, spheres):
    sc = scene(80, spheres, 2, 11, 9, 3, sky=True)
    n = sc.camera.width * sc.camera.height
    (acc, img), = reference_entry(sc, [frames], ATX_ACCEL_BVH, True)
    bufs = [DeviceArray(n * 16), DeviceArray(n * 16), DeviceArray(n * 4)]
    try:
        acc_n, img_n = noalloc(sc, 1, frames, ATX_ACCEL_BVH, True, bufs)
    finally:
        for b in bufs:
            b.free()
    assert np.array_equal(acc_n.view(np.uint32), acc.reshape(-1, 4).view(np.uint32))
    assert np.array_equal(img_n, img.reshape(-1))
