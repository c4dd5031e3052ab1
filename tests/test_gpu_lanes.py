"""Single frames marched by 2 or 4 lanes per ray (march_lanes in
pyvr_amd/csrc/hvr_rules.h) against the same frame marched by one: a counting
frame (hvr_sample_counts) always uses one lane and leaves its image in the
framebuffer, so both come from the same state.  Equal to the byte, at image
sizes around the tiles' edges and on both sides of each line of the rule, with
rays that end in the middle of a group, and with LUT entries whose alpha or
colour is not finite."""

import ctypes

import numpy as np
import pytest

import scenes

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (5, 3), (17, 9), (130, 67), (443, 443), (445, 443), (512, 512), (767, 513), (1086, 1086), (1087, 1087)]


@pytest.mark.parametrize("wh", SIZES)
@pytest.mark.parametrize("sf,nf,normals,ymax,tau", [("f32", "f32x3", True, 0.5, 0.99), ("f16", "sn8x3", True, 1.0, 0.4),
                                                    ("u8", "sn8x3", True, 0.02, 1.5), ("f32", "f32x3", False, 0.5, 0.95)])
def test_lanes_give_the_same_bytes(hip, wh, sf, nf, normals, ymax, tau):
    from pyvr_amd.datasets import blob_field, compute_normal_volume
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.volume import Volume

    w, h = wh
    data = blob_field((33, 20, 47), n_blobs=6, seed=9, noise=1e-3)
    vol = Volume(data=data, normals=compute_normal_volume(data) if normals else None, min_bounds=-scenes.BOX,
                 max_bounds=scenes.BOX)
    r = VolumeRenderer(w, h, light=scenes.standard_light(), scalar_format=sf, normal_format=nf)
    try:
        r.load_volume(vol)
        r.set_opacity_threshold(tau)
        r.set_transfer_functions(scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=w, y_max=ymax))
        r.set_camera(scenes.standard_camera(0.7, 0.4, 2.6))
        L, ctx = _lib.lib(), r.gl_manager.ctx
        lut = r.gl_manager._texture_at(r.gl_manager.program.values["transfer_function_lut"],
                                       type(r.gl_manager._units[r.gl_manager._newest_unit])).rgba.copy()
        for special in (False, True):
            if special:
                lut[40, 3], lut[60, 3], lut[90, 0], lut[120, 1] = -np.inf, np.inf, np.inf, np.nan
                _lib.check(L.hvr_set_lut(ctx, lut.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), len(lut)), "lut")
            for skip in (_lib.SKIP_OFF, _lib.SKIP_ON):
                _lib.check(L.hvr_set_empty_skip(ctx, skip), "skip")
                img = np.frombuffer(r.render(), np.uint8)
                counts = r.sample_counts()
                one = np.frombuffer(r.gl_manager.read_pixels(), np.uint8)
                assert np.array_equal(img, one), (special, skip)
                if w * h > 1000:
                    assert counts.max() > 30 and img.max() > 0
    finally:
        r.close()


@pytest.mark.parametrize("lb", [3, 4])
@pytest.mark.parametrize("sizes", [[(5, 3)], [(17, 9), (130, 67)], [(443, 443)], [(445, 443)], [(512, 512), (64, 65)],
                                   [(1086, 1086)], [(1087, 1087)], [(300, 200)] * 20])
def test_batches_of_few_rays_give_the_same_bytes(hip, sizes, lb):
    """Batches are marched by lanes by the rays of a class; a counting run by one."""
    from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", brick_log2=lb)
    try:
        vols = [DeviceBlobVolume(shape=s, n_blobs=6, seed=k, with_normals=k < 2)
                for k, s in enumerate(((33, 20, 47), (64, 64, 64), (40, 50, 30)))]   # the last: a class of its own
        ctf = scenes.c0(size=8, image=8).ctf
        for k, (w, h) in enumerate(sizes):
            b.add(vols[k % 3], scenes.standard_camera(0.7 + k, 0.4, 2.6), ctf, scenes.seeded_otf(5, seed=w, y_max=0.9), w, h,
                  opacity_threshold=(0.5, 0.99, 1.5)[k % 3])
        b.run()
        got = [b.result(i) for i in range(len(sizes))]
        b.run(count=True)
        assert got == [b.result(i) for i in range(len(sizes))]
        assert sum(int(b.counts(i).sum()) for i in range(len(sizes))) > 0
    finally:
        b.close()
