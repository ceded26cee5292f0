"""The host side of the HIP library where a HIP call fails, and the launches it
issues, on a stand-in for the HIP runtime (tests/cpp/host_errors_check.cpp):
nothing runs on a GPU."""
import os
import subprocess

import pytest

import sphinxsys_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cpp") / "host_errors_check")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-rdynamic", "-o", exe, os.path.join(ROOT, "tests", "cpp", "host_errors_check.cpp"), "-ldl"])
    return exe


@pytest.mark.parametrize("case", ["large_write", "options_error", "options_device", "regrown_lists", "tile_waves",
                                  "observers", "array_copies"])
def test_host_paths_on_the_stand_in(harness, case):
    r = subprocess.run([harness, sphinxsys_amd.LIBRARY_PATH, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
