"""The leap over transparent bricks by their clearance (pyvr_amd/csrc/
hvr_rules.h): the step bound under the sanitizers on the CPU, and on the GPU
frames that leap against frames that do not."""

import os
import shutil
import subprocess

import numpy as np
import pytest

import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_leaps_stay_inside_the_clearance(tmp_path):
    exe = tmp_path / "leap_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-ffp-contract=off", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "leap_check.cpp"), "-o", str(exe)], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "leaps ok" in res.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("lb", [3, 4])
@pytest.mark.parametrize("shape", [(7, 8, 9), (63, 64, 65), (300, 17, 40), (130, 127, 128), (200, 200, 136)])
def test_leaping_frames_equal_marched_ones(hip, shape, lb):
    """A mostly empty volume, whose bricks have every clearance: without
    skipping, with it (1, 2 and 4 lanes), counting, and batched, all to the
    byte."""
    from pyvr_amd.hip_renderer import _lib
    from pyvr_amd.hip_renderer.batch import BatchRenderer
    from pyvr_amd.hip_renderer.plain import PlainRenderer
    from pyvr_amd.volume import Volume

    rng = np.random.default_rng(sum(shape))
    data = np.zeros(shape, np.float32)
    for _ in range(6):   # a few dense specks, one of them in a corner
        c = [int(rng.integers(s)) for s in shape]
        data[tuple(slice(max(0, k - 2), k + 3) for k in c)] = rng.uniform(0.2, 1.0)
    data[0, -1, 0] = 0.7
    vol = Volume(data=data, min_bounds=np.array([-1, -0.5, 3], np.float32), max_bounds=np.array([1, 2, 5], np.float32))
    from pyvr_amd.camera import Camera

    cams = [Camera.from_spherical(target=np.array([0, 0.75, 4], np.float32), azimuth=a, elevation=e, roll=0.0, distance=d)
            for a, e, d in ((0.3, 0.2, 4.0), (2.1, -0.9, 5.0), (0.0, 0.0, 0.6))]
    ctf, otf = scenes.c0(size=8, image=8).ctf, scenes.seeded_otf(5, seed=3)
    p = PlainRenderer(scalar_format="f16", normal_format="f16x3", brick_log2=lb)
    b = BatchRenderer(scalar_format="f16", normal_format="f16x3", brick_log2=lb)
    try:
        want = []
        for cam in cams:
            for w, h in ((96, 80), (512, 500), (1100, 1080)):
                p.prepare(vol, cam, ctf, otf, w, h)
                _lib.check(hip.hvr_set_empty_skip(p.ctx, _lib.SKIP_OFF), "skip")
                ref, n = p.read(), p.sample_counts()
                _lib.check(hip.hvr_set_empty_skip(p.ctx, _lib.SKIP_ON), "skip")
                assert p.read() == ref, (cam.azimuth, w, h)
                assert np.array_equal(p.sample_counts(), n)
                if w > 500:
                    b.add(vol, cam, ctf, otf, w, h)
                    want.append((ref, n))
        b.run(count=True)
        counted = [b.result(i) for i in range(len(want))]
        counts = [b.counts(i) for i in range(len(want))]
        b.run()
        for i, (ref, n) in enumerate(want):
            assert b.result(i) == ref and counted[i] == ref and np.array_equal(counts[i], n), i
        assert any(np.frombuffer(r, np.uint8).any() for r, _ in want)
    finally:
        p.close()
        b.close()
