"""Volumes built brick by brick (k_build): the slot rule on the CPU, and the
stored values on the GPU, whatever the order the parts arrive in."""

import os
import shutil
import subprocess

import numpy as np
import pytest

import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_slots_and_voxels_are_inverse(tmp_path):
    exe = tmp_path / "slots_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "slots_check.cpp"), "-o", str(exe)], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0 and "slots ok" in res.stdout, res.stdout + res.stderr


FORMATS = [("f32", "none"), ("f16", "none"), ("u8", "none"), ("none", "f32x3"), ("none", "sn8x3"), ("none", "f16x3"),
           ("f32", "f32x3"), ("f16", "f32x3"), ("u8", "f32x3"), ("f32", "sn8x3"), ("f16", "sn8x3"), ("u8", "sn8x3"),
           ("f16", "f16x3")]


class _Context:
    def __init__(self, L, lb):
        import ctypes

        from pyvr_amd.hip_renderer import _lib

        self.L, self.ctx = L, ctypes.c_void_p()
        _lib.check(L.hvr_create(0, 8, 8, ctypes.byref(self.ctx)), "hvr_create")
        _lib.check(L.hvr_set_brick_log2(self.ctx, lb), "brick")

    def volume(self, shape, sf, nf):
        from pyvr_amd.hip_renderer.manager import _DeviceVolume

        return _DeviceVolume(self.L, self.ctx, shape, sf, nf)

    def close(self):
        self.L.hvr_destroy(self.ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("lb", [2, 3, 4])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 2), (7, 8, 9), (15, 16, 17), (33, 64, 31), (70, 5, 129)])
def test_parts_are_stored_in_any_order(hip, shape, lb):
    rng = np.random.default_rng(sum(shape) + lb)
    a, b = (rng.uniform(-0.2, 1.2, shape).astype(np.float32) for _ in range(2))
    n = rng.uniform(-1.1, 1.1, shape + (3,)).astype(np.float32)
    c = _Context(hip, lb)
    try:
        for sf, nf in FORMATS:
            has_s, has_n = sf != "none", nf != "none"
            for normals_first in (False, True):
                v = c.volume(shape, sf, nf)
                if has_n and normals_first:
                    v.upload_normals(n)
                if has_s:
                    v.upload_scalar(a)
                    v.upload_scalar(b)      # again, beside normals that are there
                if has_n and not normals_first:
                    v.upload_normals(n)
                s, m = v.download(scalar=has_s, normals=has_n)
                if has_s:
                    assert np.array_equal(s, scenes.dequant_scalar(b, sf)), (sf, nf)
                if has_n:
                    assert np.array_equal(m, scenes.dequant_normals(n, nf)), (sf, nf)
                v.destroy()
    finally:
        c.close()


@pytest.mark.gpu
def test_fields_larger_than_the_staging_buffer(hip):
    """A scalar field of 335 MB arrives in groups of brick layers."""
    shape = (1000, 1021, 82)
    data = (np.arange(np.prod(shape), dtype=np.uint32) * np.uint32(2654435761) >> 24).astype(np.float32).reshape(shape)
    data /= np.float32(255.0)
    c = _Context(hip, 3)
    try:
        v = c.volume(shape, "u8", "none")
        v.upload_scalar(data)
        s, _ = v.download()
        assert np.array_equal(s, scenes.dequant_scalar(data, "u8"))
        v.destroy()
    finally:
        c.close()


@pytest.mark.gpu
def test_a_volume_never_loaded_reads_as_zeros(hip):
    """Its memory may hold what another volume left there."""
    import ctypes

    from pyvr_amd.hip_renderer import VolumeRenderer, _lib
    from pyvr_amd.volume import Volume

    r = VolumeRenderer(64, 48, light=scenes.standard_light())
    try:
        r.load_volume(Volume(data=np.ones((40, 40, 40), np.float32), min_bounds=-scenes.BOX, max_bounds=scenes.BOX))
        r.set_camera(scenes.standard_camera())
        ctf = scenes.c0(size=8, image=8).ctf
        from pyvr_amd.transferfunctions import OpacityTransferFunction

        r.set_transfer_functions(ctf, OpacityTransferFunction([(0.0, 0.0), (0.5, 0.0), (1.0, 1.0)]))
        assert np.frombuffer(r.render(), np.uint8).any()
        m = r.gl_manager
        from pyvr_amd.hip_renderer.manager import _DeviceVolume

        for v in m._volumes:
            v.destroy()
        m._volumes, m._units = [], {k: t for k, t in m._units.items() if not hasattr(t, "volume")}
        empty = _DeviceVolume(m.L, m.ctx, (40, 40, 40), "f32", "none")
        _lib.check(m.L.hvr_bind(m.ctx, empty.handle, 0, empty.handle, 0), "hvr_bind")
        _lib.check(m.L.hvr_render_async(m.ctx), "hvr_render_async")
        assert not np.frombuffer(m.read_pixels(), np.uint8).any()
        empty.destroy()
    finally:
        r.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1024, 1023, 1), (1024, 1024, 1), (1024, 1025, 1), (1024, 1024, 3), (512, 1031, 9)])
def test_uploads_around_the_piece_size(hip, shape):
    """Pieces of 4 MiB go through three pinned parts in turn."""
    rng = np.random.default_rng(shape[1])
    c = _Context(hip, 3)
    try:
        v = c.volume(shape, "f32", "f32x3")
        for _ in range(2):
            a, n = rng.random(shape, dtype=np.float32), rng.random(shape + (3,), dtype=np.float32)
            v.upload_scalar(a)
            v.upload_normals(n)
            s, m = v.download(True, True)
            assert np.array_equal(s, a) and np.array_equal(m, n)
        v.destroy()
    finally:
        c.close()


@pytest.mark.gpu
def test_a_block_kept_from_one_volume_serves_the_next(hip):
    """Volumes of equal, slightly smaller and larger sizes after one another, in
    two contexts, and one loaded in the block of a volume released while a
    batch that reads it is in flight."""
    from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume

    rng = np.random.default_rng(5)
    one, two = _Context(hip, 3), _Context(hip, 4)
    try:
        for edge in (64, 64, 62, 40, 90, 64):
            for c in (one, two):
                shape = (edge, edge + 1, edge - 3)
                a, n = rng.random(shape, dtype=np.float32), rng.random(shape + (3,), dtype=np.float32)
                v = c.volume(shape, "f16", "f16x3")
                v.upload_normals(n)
                v.upload_scalar(a)
                s, m = v.download(True, True)
                assert np.array_equal(s, scenes.dequant_scalar(a, "f16"))
                assert np.array_equal(m, scenes.dequant_normals(n, "f16x3"))
                v.destroy()
    finally:
        one.close()
        two.close()
    b = BatchRenderer(scalar_format="f16", normal_format="f16x3")
    try:
        vols = [DeviceBlobVolume(shape=(96, 96, 96), seed=k) for k in range(3)]
        ctf, otf = scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=3)
        want = []
        for overlap in (False, True):
            for k, vol in enumerate(vols):
                for _ in range(4):
                    b.add(vol, scenes.standard_camera(0.3 * k, 0.2, 3.0), ctf, otf, 640, 640)
                slot = b.submit()
                if not overlap:
                    b.wait(slot)
                b.release(vol)
                b.upload(vols[(k + 1) % 3])
                b.wait(slot)
                img = [b.result(i, slot) for i in range(4)]
                if overlap:
                    assert img == want[k], k
                else:
                    want.append(img)
        assert want[0] != want[1] != want[2]
    finally:
        b.close()
