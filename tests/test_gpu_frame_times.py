"""What a frame's device times hold (hvr_last_kernel_ms, hvr_timing_end): the
transparent-brick flags that a LUT or volume change has the next frame
recompute are in its march time.  The flags kernel and the copy of its count
are two packets after one another on the stream, which take above 3 us; frames
of the same kind differ by less in their best of several."""

import ctypes

import numpy as np
import pytest

import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [False, True])
def test_recomputed_flags_are_in_the_march_time(hip, order):
    from pyvr_amd.config import RenderConfig
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.volume import Volume

    data = np.zeros((260, 260, 260), np.float32)
    data[::50, ::50, ::50] = 1.0
    vol = Volume(data=data, normals=np.zeros(data.shape + (3,), np.float32), min_bounds=-scenes.BOX, max_bounds=scenes.BOX)
    r = VolumeRenderer(128, 128, config=RenderConfig.preview(), light=scenes.standard_light(), scalar_format="u8",
                       normal_format="sn8x3")
    L, ctx = hip, r.gl_manager.ctx
    try:
        ctf, otf = scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=3)

        def change_lut():
            r.set_transfer_functions(ctf, otf)

        def change_volume():
            r.load_volume(vol)

        change_volume()
        change_lut()
        r.set_camera(scenes.standard_camera(0.3, 0.2, 3.0))
        _lib.check(L.hvr_set_empty_skip(ctx, _lib.SKIP_ON), "skip")
        _lib.check(L.hvr_set_dispatch_order(ctx, _lib.ORDER_ON if order else _lib.ORDER_OFF), "order")

        def frame(change=None):
            if change is not None:
                change()
            r.render()
            march, setup = r.last_kernel_ms()
            assert (setup > 0) == order
            return march

        def region(change=None):
            _lib.check(L.hvr_timing_begin(ctx, 8), "begin")
            for k in range(3):
                if change is not None and k == 1:
                    change()
                r.render()
            march, setup, n = ctypes.c_double(), ctypes.c_double(), ctypes.c_int()
            _lib.check(L.hvr_timing_end(ctx, ctypes.byref(march), ctypes.byref(setup), ctypes.byref(n)), "end")
            assert n.value == 3 and (setup.value > 0) == order
            return march.value

        for timed in (frame, region):
            timed()
            steady = min(timed() for _ in range(12))
            for change in (change_lut, change_volume):
                assert min(timed(change) for _ in range(12)) > steady + 0.003
            _lib.check(L.hvr_set_empty_skip(ctx, _lib.SKIP_OFF), "skip")
            timed(change_lut)
            _lib.check(L.hvr_set_empty_skip(ctx, _lib.SKIP_ON), "skip")
    finally:
        r.close()
