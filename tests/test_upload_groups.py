"""The groups of bricks a host field is uploaded in (upload_group,
pyvr_amd/csrc/hvr_rules.h), compiled natively and checked by
tests/native/groups_check.cpp."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_groups_hold_their_bricks_source_and_fit_the_bound(tmp_path):
    exe = tmp_path / "groups_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "pyvr_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "groups_check.cpp"), "-o", str(exe)], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    res = subprocess.run([str(exe)], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0 and "groups ok" in res.stdout, res.stdout + res.stderr
