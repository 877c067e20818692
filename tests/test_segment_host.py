"""A compiled segment's staging of small inputs and outputs without a GPU: tests/segment_host_check.cpp stands in for the
HIP runtime (two devices, streams whose work runs when something waits, a last-error slot that keeps an error until it is
read, allocations and launches that can be refused) and drives the library's segments through its C API."""
import os
import shutil
import subprocess

import pytest

from sharplight_amd import native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("g++ or the HIP headers are not available")
    native.lib()
    exe = tmp_path_factory.mktemp("segment") / "segment_host_check"
    lib = os.path.join(ROOT, "sharplight_amd")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", "-rdynamic", "-o", str(exe),
                    os.path.join(ROOT, "tests", "segment_host_check.cpp"), os.path.join(lib, "libsharplight_hip.so"), f"-Wl,-rpath,{lib}"],
                   check=True, capture_output=True, timeout=300)
    return exe


@pytest.mark.parametrize("scenario", ["close_keeps_the_error_of_another", "another_current_device", "staging_memory_refused",
                                      "failed_output_keeps_the_inputs"])
def test_segment(check, scenario):
    r = subprocess.run([str(check), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
