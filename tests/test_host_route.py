"""The rules that choose a handle's kernels, on the CPU under AddressSanitizer
and UBSan (tests/host/route_check.cpp): the expansion of the far field is not
taken where only its field layout would send the shell sums to FP64 tables in
global memory, which a captured step cannot allocate, nor by dilute systems,
whose direct sums are the faster.
"""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "gauss-legendre-spherical-t_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None or
                    not os.path.isdir("/opt/rocm/include"),
                    reason="needs g++ and the ROCm headers")
def test_routes_of_the_far_field(tmp_path):
    exe = str(tmp_path / "route_check")
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-I" + os.path.join(REPO, "include"),
         "-I" + CSRC, "-fsanitize=address,undefined",
         "-fno-sanitize-recover=undefined",
         os.path.join(REPO, "tests", "host", "route_check.cpp"),
         os.path.join(CSRC, "numerics.cpp"), "-o", exe],
        check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "failures 0" in r.stdout, r.stdout + r.stderr
