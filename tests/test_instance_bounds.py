"""Boxes of instances in the world tree, from the library's host builder
(tests/host/instance_bounds_driver.cpp)."""
import shutil
import subprocess

import pytest

from psycles_amd import build

ROOT = build.PKG.parent


def test_boxes_hold_their_instances_within_a_budget(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "instance_bounds_driver"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", f"-I{build.ROCM / 'include'}",
                    "-D__HIP_PLATFORM_AMD__", f"-I{build.CSRC}",
                    str(ROOT / "tests" / "host" / "instance_bounds_driver.cpp"), str(build.CSRC / "psx_bvh.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
