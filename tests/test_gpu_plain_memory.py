"""A plain-kernel call's device memory does not grow with its frames: 200000
frames of a tiny image in one call, equal to the same frames in calls of 50000."""
import ctypes as C

import numpy as np
import pytest

from ataraxia_amd import ATX_KERNEL_PLAIN, Renderer
from test_zz_no_alloc import _hip, scene

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_many_frames_in_one_call():
    sc = scene(91, 3, 1, 8, 8, 2)
    out = []
    for calls in ([50000] * 4, [200000]):
        print(f"case plain frames {calls}", flush=True)
        with Renderer() as r:
            r.set_kernel(ATX_KERNEL_PLAIN)
            r.on_resize(8, 8)
            r.set_settings(sc.settings)
            r.set_scene(sc)
            r.render_frames(sc.camera, 1)
            before = free_bytes()
            for n in calls:
                r.render_frames(sc.camera, n)
            grown = before - free_bytes()
            out.append((r.get_accumulation(), r.frame_index))
        assert grown < 16 << 20, grown
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1] == 200002
