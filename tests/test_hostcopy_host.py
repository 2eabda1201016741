"""Large host copies on the CPU: the library's copy code over a runtime that
counts its calls (hostcopy_driver.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "swfwi_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    cxx = shutil.which("g++")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if not cxx or not os.path.exists(os.path.join(rocm, "include", "hip", "hip_runtime.h")):
        pytest.skip("no host compiler or HIP headers")
    exe = str(tmp_path_factory.mktemp("hc") / "hostcopy_driver")
    subprocess.run([cxx, "-O1", "-g", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I",
                    os.path.join(rocm, "include"), os.path.join(HERE, "hostcopy_driver.cpp"),
                    os.path.join(CSRC, "hostcopy.cpp"), "-o", exe, "-pthread"], check=True)
    return exe


@pytest.mark.parametrize("what", ["pageable", "known", "no_pin", "no_memory"])
def test_copies(driver, what):
    """Ordinary memory goes through pinned pieces; memory that the runtime knows
    goes to it whole, and the host does not touch it.  Without pinned memory the
    runtime copies; an allocation that fails on the way (each in turn, the
    threads' own among them) ends in an exception at most."""
    subprocess.run([driver, what], check=True, timeout=60)
