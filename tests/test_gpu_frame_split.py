"""How a frame is split over the device -- the lanes per ray (march_lanes) and
the order of its blocks (row_rotation, both in pyvr_amd/csrc/hvr_rules.h) --
changes no byte of it: the frame in row order, the same frame ordered by cost
and the one-lane frame of hvr_sample_counts are equal, at image sizes on both
sides of each line of the rules for long and short rays and at row lengths
just inside and outside those that are rotated."""

import numpy as np
import pytest

import scenes

pytestmark = pytest.mark.gpu

# widths: 15 / 16 / 31 / 33 / 36 blocks of 16 rays and 28 / 35 of 8; sizes: 3/8,
# 1/2, 3/4, 7/8, 1 and 3/2 of the rays that 256 compute units hold
SIZES = [(225, 31), (248, 60), (280, 60), (490, 401), (492, 400), (512, 511), (512, 513), (528, 700), (576, 684),
         (676, 677), (678, 677), (724, 724), (725, 725), (886, 887), (888, 887)]


@pytest.mark.parametrize("wh", SIZES)
@pytest.mark.parametrize("sf,nf,step,box", [("f32", "f32x3", 0.02, 1.0), ("f16", "f16x3", 0.012, 1.0),
                                            ("u8", "sn8x3", 0.006, 1.0), ("f32", "f32x3", 0.006, 1.0)])
def test_the_split_of_a_frame_changes_no_byte(hip, wh, sf, nf, step, box):
    from pyvr_amd.config import RenderConfig
    from pyvr_amd.datasets import blob_field, compute_normal_volume
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.volume import Volume

    data = blob_field((23, 40, 31), n_blobs=6, seed=7, noise=1e-3)
    one = np.full(3, box, np.float32)
    vol = Volume(data=data, normals=compute_normal_volume(data), min_bounds=-one, max_bounds=one)
    r = VolumeRenderer(*wh, config=RenderConfig.custom(step_size=step, max_steps=1000), light=scenes.standard_light(),
                       scalar_format=sf, normal_format=nf)
    try:
        r.load_volume(vol)
        r.set_transfer_functions(scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=wh[0], y_max=0.4))
        r.set_camera(scenes.standard_camera(0.7, 0.4, 2.6))
        L, ctx = _lib.lib(), r.gl_manager.ctx
        for skip in (_lib.SKIP_OFF, _lib.SKIP_ON):
            _lib.check(L.hvr_set_empty_skip(ctx, skip), "skip")
            frames = []
            for order in (_lib.ORDER_OFF, _lib.ORDER_ON):
                _lib.check(L.hvr_set_dispatch_order(ctx, order), "order")
                frames.append(np.frombuffer(r.render(), np.uint8))
            counts = r.sample_counts()
            frames.append(np.frombuffer(r.gl_manager.read_pixels(), np.uint8))
            assert np.array_equal(frames[0], frames[1]) and np.array_equal(frames[0], frames[2]), skip
            assert counts.max() > 30 and frames[0].max() > 0
    finally:
        r.close()
