"""GPU check of what a render call counts: a trace settled by exact distances
counts once, however many spheres' orders were open."""
import pytest

from ataraxia_amd import ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT, Camera, Renderer, Settings
from ataraxia_amd.scene import FlatScene, SplitMix64, random_scene

pytestmark = pytest.mark.gpu


def stats(sc, kernel):
    print(f"case counts {sc.name} kernel={kernel}", flush=True)
    with Renderer() as r:
        r.set_kernel(kernel)
        r.on_resize(sc.camera.width, sc.camera.height)
        r.set_settings(sc.settings)
        r.set_scene(sc)
        r.render_frames(sc.camera, 1)
        return r.stats()


@pytest.mark.parametrize("kernel", [ATX_KERNEL_PLAIN, ATX_KERNEL_WAVEFRONT], ids=["plain", "wavefront"])
def test_open_traces_count_once(kernel):
    # 30 of 60 spheres in one place: the camera's rays meet all of them, at equal distances
    sph, mat, lig = random_scene(SplitMix64(62), 60, 1, 30.0, (0.0, 4.0), (10.0, 20.0), ground=False)
    sph["center"][::2] = (0.0, 1.0, 0.0)
    sph["radius"][::2] = 1.0
    cam = Camera(position=(0.0, 1.0, 1.2), direction=(0.0, 0.0, -1.0), width=40, height=24)
    st = stats(FlatScene(sph, mat, lig, Settings(True, True, 2), cam, name="one place"), kernel)
    assert st["box_tests"] > 0 and 0 < st["exact_retraces"] <= st["rays"]
