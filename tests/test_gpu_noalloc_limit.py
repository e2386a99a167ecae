"""The allocation-free call at the size from which on a scene fits its 8 MiB only
without tiles: one sphere less and one more against the renderer, bit for bit."""
import numpy as np
import pytest

from ataraxia_amd import ATX_ACCEL_BVH, Settings
from ataraxia_amd.scene import Camera, FlatScene, make_lights, make_materials, make_spheres
from test_zz_no_alloc import DeviceArray, noalloc, reference_entry

pytestmark = pytest.mark.gpu


def packed_bytes(n):
    """Spheres, material ids, one material, one light, tiles, boxes, spheres and ids by slot."""
    tiles = (n + 31) // 32
    parts = [16 * n, 4 * n, 48, 32, 2048 * tiles, 32 * (tiles + (tiles + 7) // 8), 16 * n, 4 * n]
    return sum((p + 255) // 256 * 256 for p in parts)


MOST = max(n for n in range(79000, 81000) if packed_bytes(n) <= 8 << 20)


@pytest.mark.parametrize("n", [MOST, MOST + 1])
def test_at_the_limit(n):
    rng = np.random.default_rng(5)
    sph, mat, lig = make_spheres(n), make_materials(1), make_lights(1)
    sph["center"] = rng.uniform(-40.0, 40.0, (n, 3))
    sph["radius"] = rng.uniform(0.1, 0.4, n)
    mat["albedo"][0] = (0.7, 0.6, 0.5)
    mat["roughness"][0] = 0.5
    lig["position"][0] = (0.0, 60.0, 60.0)
    lig["color"][0] = 1.0
    lig["intensity"][0] = 2000.0
    sc = FlatScene(sph, mat, lig, Settings(True, True, 2), Camera.looking_at((0.0, 10.0, 90.0), width=16, height=12),
                   name=f"limit{n}")
    (acc, img), = reference_entry(sc, [2], ATX_ACCEL_BVH, False)
    px = 16 * 12
    bufs = [DeviceArray(px * 16), DeviceArray(px * 16), DeviceArray(px * 4)]
    try:
        acc_n, img_n = noalloc(sc, 1, 2, ATX_ACCEL_BVH, False, bufs)
    finally:
        for b in bufs:
            b.free()
    assert np.array_equal(acc_n.view(np.uint32), acc.reshape(-1, 4).view(np.uint32))
    assert np.array_equal(img_n, img.reshape(-1)) and np.ptp(acc_n[:, 0]) > 0
