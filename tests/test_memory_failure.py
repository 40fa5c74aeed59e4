"""Host code of the library when device memory runs out, on a pretended device
(tests/host/memory_failure_driver.cpp): what a failed call leaves behind is
never handed to a kernel, and later calls work again."""
import shutil
import subprocess

import pytest

from psycles_amd import build

ROOT = build.PKG.parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("memory") / "memory_failure_driver"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{build.ROCM / 'include'}", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROOT / 'include'}", f"-I{build.CSRC}", str(ROOT / "tests" / "host" / "memory_failure_driver.cpp"),
                    "-o", str(exe), "-rdynamic", f"-L{build.PKG}", "-lpsx", f"-Wl,-rpath,{build.PKG}",
                    f"-Wl,-rpath,{build.ROCM / 'lib'}"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["table", "path-state", "film", "passes", "broken", "parameters"])
def test_after_a_failed_allocation(driver, scenario):
    r = subprocess.run([str(driver), scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
