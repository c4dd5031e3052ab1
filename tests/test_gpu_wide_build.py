"""Volumes built with 64-bit voxel offsets (k_build from 2^30 voxels on;
HVR_BUILD=wide for every volume) against those built with 32-bit ones: the
stored fields bit for bit, and a frame whose samples read the aprons, from
host fields, from a field with its normals and from generated blobs, over equal
and unequal axes, bricks at the faces and clear of them, through the caches and
past them."""

import numpy as np
import pytest

import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lb", [3, 4])
@pytest.mark.parametrize("shape,formats", [((2, 2, 2), [("f32", "f32x3")]),
                                           ((33, 20, 33), [("f32", "f32x3"), ("f16", "f16x3"), ("u8", "sn8x3")]),
                                           ((33, 64, 31), [("f32", "f32x3"), ("f16", "sn8x3"), ("u8", "f32x3")]),
                                           ((50, 35, 50), [("f16", "f32x3"), ("f32", "sn8x3")]),
                                           ((240, 232, 240), [("f32", "f32x3")])])   # 320 MB of texels
def test_wide_offsets_build_the_same_volume(hip, monkeypatch, shape, formats, lb):
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.hip_renderer.manager import _DeviceVolume
    from pyvr_amd.volume import Volume

    rng = np.random.default_rng(sum(shape) + lb)
    data = rng.random(shape, dtype=np.float32)
    normals = rng.uniform(-1.0, 1.0, shape + (3,)).astype(np.float32)

    def results(sf, nf):
        r = VolumeRenderer(96, 80, light=scenes.standard_light(), scalar_format=sf, normal_format=nf)
        m = r.gl_manager
        try:
            _lib.check(hip.hvr_set_brick_log2(m.ctx, lb), "brick")
            r.set_camera(scenes.standard_camera(0.7, 0.4, 2.6))
            r.set_transfer_functions(scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=2, y_max=0.05))
            r.load_volume(Volume(data=data, normals=normals, min_bounds=-scenes.BOX, max_bounds=scenes.BOX))
            out = [r.render()]
            v = _DeviceVolume(hip, m.ctx, shape, sf, nf)
            loads = [lambda: (v.upload_normals(normals), v.upload_scalar(data)), lambda: v.upload_scalar_normals(data),
                     lambda: v.generate_blobs([[0.1, -0.2, 0.3], [-0.5, 0.4, 0.0]], [0.3, 0.2], [0.7, 0.9], 1e-3, 5)]
            for load in loads:
                load()
                out.extend(a.tobytes() for a in v.download(True, True))
                _lib.check(hip.hvr_bind(m.ctx, v.handle, 0, v.handle, 1), "hvr_bind")
                _lib.check(hip.hvr_render_async(m.ctx), "hvr_render_async")
                out.append(m.read_pixels())
            v.destroy()
            return out
        finally:
            r.close()

    for sf, nf in formats:
        monkeypatch.delenv("HVR_BUILD", raising=False)
        want = results(sf, nf)
        monkeypatch.setenv("HVR_BUILD", "wide")
        got = results(sf, nf)
        assert [a == b for a, b in zip(want, got)] == [True] * 10, (sf, nf)
        assert np.frombuffer(want[0], np.uint8).any()
