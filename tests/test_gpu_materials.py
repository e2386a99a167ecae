"""GPU check of the shading's quotients at the ends of the materials' ranges:
accumulations equal the oracle's bit for bit where the short forms apply, where
one operand sends a lane to the general form, and for scenes outside the
ranges."""
import numpy as np
import pytest

from _scenes import oracle_accumulate
from ataraxia_amd import ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT, Camera, Renderer, Settings
from ataraxia_amd.scene import FlatScene, SplitMix64, random_scene

pytestmark = pytest.mark.gpu

CASES = {
    "zeros": dict(albedo=(0.0, 0.8, 0.0), roughness=0.0, metallic=0.0),       # black channels, a2 = 0
    "black": dict(albedo=(0.0, 0.0, 0.0), roughness=1.0, metallic=1.0),       # throughput 0, F = (1 - cos)^5
    "ones": dict(albedo=(1.0, 1.0, 1.0), F0=(1.0, 1.0, 1.0), roughness=1.0, metallic=1.0),
    "smooth": dict(roughness=2.0 ** -10, metallic=1.0),                       # a2 = 2^-40
    "smoother": dict(roughness=2.0 ** -11, metallic=0.5),                     # outside: the general forms
    "dim": dict(albedo=(2.0 ** -13, 0.5, 1.0)),                               # 2^-78 after 6 bounces
    "dimmer": dict(albedo=(2.0 ** -14, 0.5, 1.0)),                            # outside
    "bright": dict(albedo=(1.5, 0.5, 1.0)),                                   # outside
    "tiny F0": dict(F0=(0.0, 2.0 ** -120, 1.0), metallic=0.0),
}


@pytest.mark.parametrize("kernel", [ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT], ids=["plain", "wavefront"])
@pytest.mark.parametrize("name", list(CASES))
def test_material_ranges(name, kernel):
    print(f"case materials {name} kernel={kernel}", flush=True)
    sph, mat, lig = random_scene(SplitMix64(11), 40, 2, 9.0, (0.0, 4.0), (10.0, 20.0))
    for k, v in CASES[name].items():
        mat[k][::2] = v
    cam = Camera.looking_at((0.0, 4.0, 18.0), width=67, height=45)
    sc = FlatScene(sph, mat, lig, Settings(True, True, 6), cam, name="materials")
    with Renderer() as r:
        r.set_kernel(kernel)
        r.on_resize(cam.width, cam.height)
        r.set_settings(sc.settings)
        r.set_scene(sc)
        r.render_frames(cam, 4)
        acc = r.get_accumulation().reshape(-1, 4)
    assert np.array_equal(acc, oracle_accumulate(sc, 4)[0], equal_nan=True)
