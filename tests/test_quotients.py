"""Quotients of a gradient's components by one reciprocal (put_gradient,
pyvr_amd/csrc/hvr_device.h): correctly rounded for every divisor mantissa, on
the CPU from every approximation a reciprocal instruction within an ulp may
give, and on the GPU from the one it gives."""

import os
import shutil
import subprocess

import numpy as np
import pytest

from test_build import _Context

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_divisor_mantissa_and_every_seed(tmp_path):
    exe = tmp_path / "quotient_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "quotient_check.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and "quotients ok" in res.stdout, res.stdout + res.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("part", range(8))
def test_every_divisor_mantissa_on_the_device(hip, part):
    """Gradients (d, 0, 2^-23) with every mantissa of d in [1, 2): the norm is d
    (the other square and 1e-8 are below half its ulp) or, where the square root
    rounds the other way, a neighbour of it, which the first component tells
    (d / d = 1 and no other quotient of neighbours is)."""
    n = 1 << 20
    d = np.float32(1) + (np.arange(n, dtype=np.float32) + np.float32(part * n)) * np.float32(2.0 ** -23)
    f = np.zeros((2, 2, n), np.float32)
    f[1] = d
    c = _Context(hip, 3)
    try:
        v = c.volume(f.shape, "f32", "f32x3")
        v.upload_scalar_normals(f)
        _, normals = v.download(scalar=False, normals=True)
        got = normals.reshape(2, 2, n, 3)[1, 0]
        plain = got[:, 0] == 1
        assert plain.mean() > 0.5
        assert np.array_equal(got[plain, 2], (np.float32(2.0 ** -23) / d)[plain])
        assert np.all(got[:, 1] == 0)
        v.destroy()
    finally:
        c.close()
