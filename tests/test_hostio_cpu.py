"""The host side of the transfers (slgpu_hostio.h), compiled for the CPU against a HIP runtime of a few
lines (tests/cpp/hostio_check.cpp): bytes arrive whole, the time from the last device copy until the
caller's arrays are filled is reported, which the phase timers add to their events' time, and the copying
threads are no more than the cores the process may use beside the caller's."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("no g++ or no HIP headers")
    exe = str(tmp_path_factory.mktemp("hostio") / "hostio_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                        os.path.join(HERE, "cpp", "hostio_check.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_outputs(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
