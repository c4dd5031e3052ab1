"""Which way an upload takes (upload_host in pyvr_amd/csrc/hipvr.hip): pageable
host memory through the library's pinned ring, memory the device can read by
itself straight, whatever part of it the caller passes; and the groups of
bricks a field arrives in (upload_group in pyvr_amd/csrc/hvr_rules.h)."""

import numpy as np
import pytest

from test_build import _Context

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def disarm():
    from pyvr_amd.hip_renderer import _lib

    yield
    _lib.inject_fault(None)


@pytest.mark.parametrize("pinned,offset,takes_ring", [(False, 0, True), (True, 0, False), (True, 4096, False),
                                                      (True, 4, False)])
def test_pinned_data_is_copied_straight(hip, pinned, offset, takes_ring):
    import ctypes

    from pyvr_amd.hip_renderer import _lib

    shape = (130, 120, 110)   # 6.9 MB, above the ring's 4 MiB pieces
    n = int(np.prod(shape))
    c = _Context(hip, 3)
    frame = ctypes.c_void_p()
    _lib.check(hip.hvr_create(0, 2048, 1024, ctypes.byref(frame)), "hvr_create")
    try:
        if pinned:   # a frame's pinned pixels, 8 MiB
            _lib.check(hip.hvr_render_async(frame), "render")
            ptr = ctypes.POINTER(ctypes.c_uint8)()
            _lib.check(hip.hvr_read_pinned(frame, ctypes.byref(ptr)), "read")
            pool = np.ctypeslib.as_array(ptr, shape=(2048 * 1024 * 4,)).view(np.float32)
        else:
            pool = np.empty(n + 1024, np.float32)
        a = pool[offset // 4:offset // 4 + n].reshape(shape)
        a[...] = np.random.default_rng(3).random(shape, dtype=np.float32)
        v = c.volume(shape, "f32", "f32x3")
        v.upload_scalar(a)
        assert np.array_equal(v.download()[0], a)
        for upload in (v.upload_scalar, v.upload_scalar_normals):
            _lib.inject_fault("hvr_upload_ring", code=-2)
            if takes_ring:
                with pytest.raises(RuntimeError, match="injected fault in hvr_upload_ring"):
                    upload(a)
            else:
                upload(a)
        _lib.inject_fault(None)
        v.upload_scalar_normals(a)          # and again after the failures
        assert np.array_equal(v.download()[0], a)
        v.destroy()
    finally:
        c.close()
        hip.hvr_destroy(frame)


@pytest.mark.parametrize("lb", [3, 4])
def test_large_planes_stay_within_the_staging_bound(hip, lb):
    """Planes of 50 MB of normals: 9 or 17 of them would be 450 or 850 MB.  What the
    context keeps after the volume is gone is the staging buffer."""
    from pyvr_amd.hip_renderer import _lib

    def used():
        free, total = _lib.device_memory(0)
        return total - free

    shape = (2048, 2048, 20)
    rng = np.random.default_rng(lb)
    normals = rng.integers(-127, 128, (2048, 1, 20, 3), dtype=np.int8) / np.float32(127)
    normals = np.broadcast_to(normals, shape + (3,)) * np.linspace(-1, 1, 2048, dtype=np.float32)[None, :, None, None]
    normals = np.ascontiguousarray(normals, dtype=np.float32)
    c = _Context(hip, lb)
    try:
        before = used()
        v = c.volume(shape, "none", "f32x3")     # above what a destroyed volume leaves for the next
        v.upload_normals(normals)
        assert np.array_equal(v.download(scalar=False, normals=True)[1], normals)
        v.destroy()
        assert used() - before <= (256 << 20) + (8 << 20)
    finally:
        c.close()


@pytest.mark.parametrize("lb", [3, 4])
@pytest.mark.parametrize("stage", [400000, 200000, 100000, 1000])
@pytest.mark.parametrize("sf,nf", [("f32", "f32x3"), ("f16", "f16x3"), ("u8", "sn8x3")])
def test_groups_of_bricks_build_the_same_volume(hip, monkeypatch, stage, lb, sf, nf):
    """Groups of layers and of rows of one layer (both fields, the second beside the
    first): the stored fields, and a frame whose samples read the aprons."""
    import scenes
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.hip_renderer.manager import _DeviceVolume
    from pyvr_amd.volume import Volume

    shape = (70, 45, 129)
    rng = np.random.default_rng(stage + lb)
    data = rng.random(shape, dtype=np.float32)
    normals = rng.uniform(-1.0, 1.0, shape + (3,)).astype(np.float32)
    vol = Volume(data=data, normals=normals, min_bounds=-scenes.BOX, max_bounds=scenes.BOX)

    def renderer():
        r = VolumeRenderer(160, 120, light=scenes.standard_light(), scalar_format=sf, normal_format=nf)
        _lib.check(hip.hvr_set_brick_log2(r.gl_manager.ctx, lb), "brick")
        r.set_camera(scenes.standard_camera(0.7, 0.4, 2.6))
        r.set_transfer_functions(scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=2, y_max=0.05))
        r.load_volume(vol)
        return r

    whole = renderer()
    monkeypatch.setenv("HVR_STAGE", str(stage))
    parts = renderer()
    try:
        want = whole.render()
        assert np.frombuffer(want, np.uint8).max() > 0
        assert parts.render() == want
        m = parts.gl_manager
        for normals_first in (False, True):
            v = _DeviceVolume(hip, m.ctx, shape, sf, nf)
            if normals_first:
                v.upload_normals(normals)
            v.upload_scalar(1.0 - data)
            v.upload_scalar(data)
            if not normals_first:
                v.upload_normals(normals)
            s, n = v.download(True, True)
            assert np.array_equal(s, scenes.dequant_scalar(data, sf)) and np.array_equal(n, scenes.dequant_normals(normals, nf))
            _lib.check(hip.hvr_bind(m.ctx, v.handle, 0, v.handle, 1), "hvr_bind")
            _lib.check(hip.hvr_render_async(m.ctx), "hvr_render_async")
            assert m.read_pixels() == want
            v.destroy()
    finally:
        whole.close()
        parts.close()
