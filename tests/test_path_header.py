"""Parts of the device header psx_path.h by themselves.

The short reciprocal, root and quotient of the light importance: on the host
for every approximation that the hardware may give, on the device for those it
gives.  The traversal stack's bookkeeping, on the host."""
import shutil
import subprocess

import pytest

from psycles_amd import build

ROOT = build.PKG.parent
CLANG = build.ROCM / "llvm" / "bin" / "clang++"


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which(str(CLANG)) is None:
        pytest.skip("clang++ not available")
    exe = tmp_path_factory.mktemp("header") / "path_header_driver"
    subprocess.run([str(CLANG), "-x", "c++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-Wno-unused-function",
                    "-Wno-unknown-attributes", f"-I{build.CSRC}", str(ROOT / "tests" / "host" / "path_header_driver.cpp"),
                    "-pthread", "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("part", ["reciprocal", "root", "quotient", "stack"])
def test_on_the_host(driver, part):
    r = subprocess.run([str(driver), part], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


@pytest.mark.gpu
def test_short_operations_on_the_device():
    exe = build.BUILD / "short_operations"
    if not exe.exists():
        exe = build.build_short_operations()
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
