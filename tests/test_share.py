"""Requests of a batch that share a volume and a LUT (pyvr_amd/csrc/
hvr_share.h): the search on the CPU, and batches that mix shared and own LUTs
on the GPU against single frames."""

import os
import shutil
import subprocess

import pytest

import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_the_search_compares_only_equal_hashes(tmp_path):
    exe = tmp_path / "share_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "share_check.cpp"), "-o", str(exe)], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0 and "share ok" in res.stdout, res.stdout + res.stderr


@pytest.mark.gpu
def test_shared_and_own_luts_in_one_batch(hip):
    """Two volumes of one and one of another class, three LUTs of two lengths: what
    is shared, and what only looks alike, renders as alone."""
    from pyvr_amd.hip_renderer.batch import BatchRenderer, DeviceBlobVolume

    b = BatchRenderer(scalar_format="f16", normal_format="f16x3")
    try:
        vols = [DeviceBlobVolume(shape=(40, 30, 50), seed=k, with_normals=k < 2) for k in range(3)]
        ctf = scenes.c0(size=8, image=8).ctf
        otfs = [scenes.seeded_otf(5, seed=s, y_max=0.6) for s in (1, 2)]
        asks = [(vols[k % 3], otfs[k // 3 % 2], (256, 256, 300)[k // 6 % 3], 0.3 * k) for k in range(24)]

        def add(ask):
            vol, otf, size, az = ask
            b.add(vol, scenes.standard_camera(az, 0.2, 3.0), ctf, otf, 48, 40, lut_size=size)

        want = []
        for ask in asks:
            b.clear()
            add(ask)
            b.run()
            want.append(b.result(0))
        b.clear()
        for ask in asks:
            add(ask)
        b.run()
        assert [b.result(k) for k in range(len(asks))] == want
        assert len(set(want)) == len(asks)
    finally:
        b.close()
