"""GPU check of the chunk queue's counters: on a grid of few waves every wave
goes on from its own counter to all the others, back to earlier scenes of the
launch; every path runs once (accumulations equal the oracle's)."""
import numpy as np
import pytest

from _scenes import oracle_accumulate
from ataraxia_amd import Batch, Camera, Settings
from ataraxia_amd.scene import FlatScene, SplitMix64, random_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spheres", [5, 40], ids=["flat", "tiles"])
@pytest.mark.parametrize("workgroups", [1, 3, 5, 64])
def test_every_chunk_runs_once(workgroups, spheres):
    print(f"case queue workgroups={workgroups} spheres={spheres}", flush=True)
    scenes = []
    # one pixel, less and more than a chunk of 64 jobs, an open sky (short hit list)
    for k, (w, h) in enumerate([(1, 1), (7, 5), (40, 23), (16, 4), (33, 31), (64, 1), (25, 16)]):
        sph, mat, lig = random_scene(SplitMix64(90 + k), spheres, 2, 9.0, (0.0, 4.0), (10.0, 20.0), ground=k % 2 == 0)
        cam = Camera.looking_at((0.0, 4.0, 18.0), width=w, height=h)
        scenes.append(FlatScene(sph, mat, lig, Settings(True, True, 4), cam, spp=5))
    with Batch() as b:
        b.set_tuning(chunk_px=64, workgroups=workgroups)
        ids = [b.add_scene(s) for s in scenes]
        b.render()
        got = [b.get_accumulation(i).reshape(-1, 4) for i in ids]
        assert b.stats()["samples"] == 5 * sum(s.camera.width * s.camera.height for s in scenes)
    for s, acc in zip(scenes, got):
        assert np.array_equal(acc, oracle_accumulate(s, 5)[0])
