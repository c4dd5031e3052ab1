"""How a frame is split over the device: the rules (pyvr_amd/csrc/hvr_rules.h)
on the CPU, and what HVR_ORDER_AUTO does for frames of one and of two lanes per
ray on the GPU.  hvr_dispatch_order_info speaks of the last frame, a counting
one included (which always has one lane), so it is read right after the
render."""

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_rules_on_both_sides_of_their_lines(tmp_path):
    exe = tmp_path / "split_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "split_check.cpp"), "-o", str(exe)], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0 and "split ok" in res.stdout, res.stdout + res.stderr


# 2 and 2.32 times the rays of 256 compute units, 8-byte texels of a small volume:
# one lane without skipping, two with it up to 2.25 times; steps: the box's
# diagonal 2 sqrt(3) over the step
@pytest.mark.gpu
@pytest.mark.parametrize("size,skip,step,expect,counting", [(1024, False, 0.01, 1, 1), (1104, False, 0.01, 1, 1),
                                                            (1104, False, 0.02, 0, 0), (1024, True, 0.005, 1, 1),
                                                            (1024, True, 0.01, 0, 1), (1104, True, 0.005, 0, 0)])
def test_auto_orders_by_the_rendered_frames_lanes(hip, size, skip, step, expect, counting):
    from pyvr_amd.config import RenderConfig
    from pyvr_amd.hip_renderer import VolumeRenderer, _lib

    sc = scenes.c0(size=48, image=64)
    r = VolumeRenderer(size, size, config=RenderConfig.custom(step_size=step, max_steps=1000), light=sc.light,
                       scalar_format="f16", normal_format="f16x3")
    L, ctx = hip, r.gl_manager.ctx

    def ordered():
        used = ctypes.c_int()
        _lib.check(L.hvr_dispatch_order_info(ctx, ctypes.byref(used)), "order info")
        return used.value

    try:
        r.load_volume(sc.volume())
        r.set_transfer_functions(sc.ctf, sc.otf, sc.lut_size)
        r.set_camera(sc.camera)
        _lib.check(L.hvr_set_empty_skip(ctx, _lib.SKIP_ON if skip else _lib.SKIP_OFF), "skip")
        img = r.render()
        assert ordered() == expect
        r.sample_counts()
        assert ordered() == counting      # the counting frame's: one lane
        _lib.check(L.hvr_set_dispatch_order(ctx, _lib.ORDER_OFF), "order")
        assert r.render() == img and ordered() == 0
        assert np.frombuffer(img, np.uint8).any()
    finally:
        r.close()
