"""Which way an upload takes (upload_host in pyvr_amd/csrc/hipvr.hip): pageable
host memory through the library's pinned ring, memory the device can read by
itself straight, whatever part of it the caller passes."""

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
