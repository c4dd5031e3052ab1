"""Memory kept between volumes: what the server's budget leaves for it (on the
CPU, with a stand-in backend), and that it is counted and given back (on the
GPU)."""

from types import SimpleNamespace

import numpy as np
import pytest

from test_serve_logic import B16, FakeBackend, vol
from pyvr_amd.hip_renderer.serve import RenderServer, batch_pool_bytes, volume_bricks


class KeepingBackend(FakeBackend):
    """Keeps the last released volume's bytes and some staging after uploads."""

    def __init__(self, staging):
        super().__init__(2)
        self.staging, self.staged, self.spare, self.trims = staging, 0, 0, 0

    def upload(self, v, device_normals=False):
        super().upload(v, device_normals)
        self.spare, self.staged = 0, self.staging     # the block serves the upload

    def release(self, v):
        super().release(v)
        self.spare = B16

    def kept_bytes(self):
        return self.spare + self.staged

    def trim(self):
        self.spare = self.staged = 0
        self.trims += 1


def _server(room, staging):
    be = KeepingBackend(staging)
    pools = 2 * batch_pool_bytes(4, 1 << 12, volume_bricks((16,) * 3))
    srv = RenderServer(backend=be, memory_budget=pools + room, pipeline=2, max_batch_requests=4, max_batch_pixels=1 << 12)
    return srv, be, pools


@pytest.mark.parametrize("staging", [0, 100, B16])
def test_the_budget_holds_with_what_is_kept(staging):
    srv, be, pools = _server(2 * B16 + 50, staging)
    for k in "ABCD":
        srv.register(k, vol(k, 16))
    for k in "ABCDABDC":
        assert srv._make_resident(k)
        assert srv.resident_bytes() + be.kept_bytes() + pools <= srv.memory_budget
    assert srv.evictions > 0
    assert (be.trims > 0) == (staging > 50)
    # D evicted for a larger volume, and still no room beside C: its block does not stay either
    srv.register("E", SimpleNamespace(name="E", data=np.zeros((16, 16, 24), np.float32), has_normals=True))
    srv._resident["C"].pins = 1
    assert not srv._make_resident("E") and srv.resident_keys() == ["C"]
    assert srv.resident_bytes() + be.kept_bytes() + pools <= srv.memory_budget


def test_kept_memory_stays_where_there_is_room():
    srv, be, _ = _server(4 * B16 + 50, B16)
    for k in "AB":
        srv.register(k, vol(k, 16))
        assert srv._make_resident(k)
    assert be.kept_bytes() == B16 and be.trims == 0


def _free():
    from pyvr_amd.hip_renderer import _lib

    return _lib.device_memory(0)[0]


SLACK = 8 << 20   # the runtime's own allocations between two looks


@pytest.mark.gpu
def test_a_released_volume_counts_as_free_and_is_given_back(hip):
    from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3")
    try:
        b.trim()
        free = _free()
        v = DeviceBlobVolume(shape=(320, 320, 320))
        nbytes = b.upload(v).nbytes()
        stage = b.kept_bytes()          # what its field passed through
        assert 4 * 320 ** 3 <= stage <= 256 << 20
        b.release(v)
        assert nbytes <= b.kept_bytes() - stage <= nbytes + nbytes // 32
        assert abs(free - stage - _free()) <= SLACK
        b.trim()
        assert b.kept_bytes() == 0 and abs(free - _free()) <= SLACK
        b.upload(v)                     # and it goes on
        b.release(v)
    finally:
        b.close()


@pytest.mark.gpu
def test_trimming_a_renderer_keeps_its_volume(hip):
    import scenes
    from pyvr_amd.hip_renderer import VolumeRenderer

    sc = scenes.c0(size=48, image=96)
    r = VolumeRenderer(sc.width, sc.height, config=sc.config, light=sc.light)
    try:
        r.load_volume(sc.volume())
        r.set_camera(sc.camera)
        r.set_transfer_functions(sc.ctf, sc.otf, sc.lut_size)
        want = r.render()
        r.trim()
        assert r.render() == want
        r.load_volume(sc.volume())
        assert r.render() == want and np.frombuffer(want, np.uint8).any()
    finally:
        r.close()
