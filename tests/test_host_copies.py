"""The large host copies (solar_amd/csrc/solar_hostcopy.cpp) on the CPU, against
a stand-in of the HIP runtime (tests/native/hip_stub.hpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "solar_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hostcopy") / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, "-I",
                    NATIVE, os.path.join(NATIVE, "host_copy_check.cpp"), os.path.join(CSRC, "solar_hostcopy.cpp"),
                    "-pthread", "-o", out], check=True)
    return out


@pytest.mark.parametrize("case", ["other_device", "known_memory", "events_fail", "no_thread", "two_threads", "settled_stream", "first_copy"])
def test_host_copy(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
