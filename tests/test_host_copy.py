"""The host part of the state transfers (dgtd_amd/csrc/host_copy.cpp) on the
CPU: tests/cpp/host_copy_check.cpp runs it over a stand-in for the HIP calls
whose copies complete late."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dgtd_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_copy") / "host_copy_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(HERE, "cpp", "host_copy_check.cpp"), os.path.join(CSRC, "host_copy.cpp")], check=True)
    return exe


@pytest.mark.parametrize("test", ["round_trips", "failing_allocations", "failing_copies", "no_pinned_memory", "threads",
                                  "pinned_memory"])
def test_host_copy(program, test):
    r = subprocess.run([program, test], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.endswith("OK\n")
