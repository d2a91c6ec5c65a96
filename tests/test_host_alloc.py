"""What handles and batches allocate, with their host code run on the CPU
against a stand-in for the HIP runtime that limits and tracks device memory
(tests/host/fake_hip.hpp, alloc_check.cpp), under AddressSanitizer and UBSan.
"""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "gauss-legendre-spherical-t_amd", "csrc")


@pytest.fixture(scope="module")
def alloc_check(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the ROCm headers")
    exe = str(tmp_path_factory.mktemp("alloc") / "alloc_check")
    src = [os.path.join(REPO, "tests", "host", "alloc_check.cpp")] + [
        os.path.join(CSRC, f) for f in ("engine.hip", "batch.hip",
                                        "numerics.cpp")]
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-I" + os.path.join(REPO, "include"),
         "-I" + CSRC, "-fsanitize=address,undefined",
         "-fno-sanitize-recover=undefined", "-x", "c++", *src, "-o", exe],
        check=True, timeout=300)
    return exe


@pytest.mark.parametrize("what", ["handle", "capture", "batch", "slots", "layout",
                                  "tune"])
def test_allocations(alloc_check, what):
    r = subprocess.run([alloc_check, what], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
