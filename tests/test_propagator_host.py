"""What the propagator decides on the host, on the CPU: its own sources over
launchers that count (propagator_driver.cpp)."""
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
    exe = str(tmp_path_factory.mktemp("prop") / "propagator_driver")
    subprocess.run([cxx, "-O1", "-g", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I",
                    os.path.join(rocm, "include"), os.path.join(HERE, "propagator_driver.cpp"),
                    os.path.join(CSRC, "propagator.cpp"), os.path.join(CSRC, "resident.cpp"), "-o", exe, "-pthread"],
                   check=True)
    return exe


def run(driver, what):
    r = subprocess.run([driver, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_widths_are_timed_after_a_resident_run(driver):
    """A run that takes the resident loop keeps the rule's widths as they are,
    and the first per-step run of the size still times them."""
    run(driver, "tuner")


def test_backward_widths_are_timed_for_a_backward_run(driver):
    """No trials of the backward kernel where no backward run follows, or where
    it takes the resident loop."""
    run(driver, "backward_trials")


def test_no_memory_for_the_resident_loop(driver):
    """Where its buffers cannot be had the per-step kernels run, and the resident
    loop again once there is memory."""
    run(driver, "no_memory")


def test_a_shared_chip_is_tried_again(driver):
    """After a wait that ran out a handle goes back to the resident loop: 64
    forward runs later, and after twice as many each time it is in vain again."""
    run(driver, "shared_chip")


def test_the_wait_limit(driver):
    """Finite, not negative, ten seconds at most."""
    run(driver, "wait_limit")


def test_a_few_steps_run_per_step(driver):
    """A run of fewer than 5 steps is not worth a resident launch."""
    run(driver, "few_steps")


def test_parts_only_where_they_pay(driver):
    """A batch goes as several resident launches only where that is faster than
    a launch a step, however well its tiles of 62 z are filled."""
    run(driver, "parts")
