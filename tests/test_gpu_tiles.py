"""GPU parity of the tile queries at the sizes where a tile (32 spheres), a
round of eight tiles or the groups' boxes (more than 16 tiles) begin and end:
accumulation and image equal the oracle's flat loop bit for bit."""
import numpy as np
import pytest

from _scenes import oracle_accumulate
from ataraxia_amd import ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT, Camera, Renderer, Settings
from ataraxia_amd.scene import FlatScene, SplitMix64, random_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT], ids=["plain", "wavefront"])
@pytest.mark.parametrize("spheres,ground", [(16, False), (31, True), (32, True), (33, False), (65, True), (255, False),
                                            (257, True), (512, True), (513, False), (545, True), (2049, True), (17000, True)])
def test_tile_sizes_match_oracle(spheres, ground, kernel):
    ext = 20.0 * (spheres / 256.0) ** 0.5
    sph, mat, lig = random_scene(SplitMix64(spheres), spheres, 3, ext, (0.0, 6.0), (10.0, 20.0), ground=ground)
    # the last spheres repeat the first ones: equal distances, the lower index wins
    sph["center"][-4:], sph["radius"][-4:] = sph["center"][4:8], sph["radius"][4:8]
    # an odd size leaves lanes of the last waves without a pixel
    cam = Camera.looking_at((0.0, 0.4 * ext, 2.0 * ext), width=61, height=35)
    sc = FlatScene(sph, mat, lig, Settings(True, True, 6), cam, name="tiles")
    print(f"case tiles spheres={spheres} ground={ground} kernel={kernel}", flush=True)
    with Renderer() as r:
        r.set_kernel(kernel)
        r.on_resize(cam.width, cam.height)
        r.set_settings(sc.settings)
        r.set_scene(sc)
        r.render_frames(cam, 3)
        acc, img = r.get_accumulation().reshape(-1, 4), r.get_image().reshape(-1)
    oacc, oimg = oracle_accumulate(sc, 3)
    assert np.array_equal(acc, oacc)
    assert np.array_equal(img, oimg)
