"""GPU check of the result copies: images and accumulations of sizes around
the staged copy's parts (1 MiB, four in flight) equal what the runtime copies
into pinned memory, also for callers in several threads, and a served request
returns the same."""
import ctypes
import threading

import numpy as np
import pytest

from ataraxia_amd import Camera, Renderer, Server, Settings, _lib
from ataraxia_amd.scene import FlatScene, SplitMix64, random_scene

pytestmark = pytest.mark.gpu

_hip = ctypes.CDLL("libamdhip64.so")
_hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
_hip.hipHostFree.argtypes = [ctypes.c_void_p]


@pytest.mark.parametrize("w,h", [(1, 1), (511, 513), (512, 512), (512, 513), (1024, 1024), (1031, 1027), (1920, 1081)])
def test_result_copies(w, h):
    print(f"case results {w}x{h}", flush=True)
    sph, mat, lig = random_scene(SplitMix64(7), 24, 1, 9.0, (0.0, 4.0), (10.0, 20.0))
    cam = Camera.looking_at((0.0, 4.0, 18.0), width=w, height=h)
    sc = FlatScene(sph, mat, lig, Settings(True, True, 2), cam, spp=2)
    with Renderer() as r:
        r.on_resize(w, h)
        r.set_settings(sc.settings)
        r.set_scene(sc)
        r.render_frames(cam, 2)
        pinned = ctypes.c_void_p()
        assert _hip.hipHostMalloc(ctypes.byref(pinned), w * h * 16, 0) == 0
        try:
            _lib.check(_lib.lib.atx_renderer_get_image(r._h, pinned, w * h))
            img = np.frombuffer(ctypes.string_at(pinned, w * h * 4), np.uint32)
            _lib.check(_lib.lib.atx_renderer_get_accumulation(r._h, pinned, w * h * 4))
            acc = np.frombuffer(ctypes.string_at(pinned, w * h * 16), np.float32)
        finally:
            _hip.hipHostFree(pinned)
        assert np.array_equal(r.get_image().reshape(-1), img)
        got = [None] * 3
        ts = [threading.Thread(target=lambda k=k: got.__setitem__(k, r.get_accumulation())) for k in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert all(np.array_equal(g.reshape(-1), acc) for g in got)
    with Server() as srv:
        rid = srv.submit(sc)
        srv.wait(rid)
        simg, sacc = srv.result(rid, release=True)
    assert np.array_equal(simg.reshape(-1), img) and np.array_equal(sacc.reshape(-1), acc)
