"""The far field's harmonic tables (harmonic_plan.hpp) on the CPU, under
AddressSanitizer and UBSan: plane waves put together from the tables against
cos and sin of the phase (tests/host/harm_check.cpp).

The truncation bound is 3e-7 (mixed) and 1e-15 (FP64) per wave; the check runs
in FP64, whose rounding over the recurrences (up to 56 degrees, values up to
one) stays under 1e-12.
"""
import os
import re
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "gauss-legendre-spherical-t_amd", "csrc")


@pytest.fixture(scope="module")
def harm_check(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the ROCm headers")
    exe = str(tmp_path_factory.mktemp("harm") / "harm_check")
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-I" + os.path.join(REPO, "include"),
         "-I" + CSRC, "-fsanitize=address,undefined",
         "-fno-sanitize-recover=undefined",
         os.path.join(REPO, "tests", "host", "harm_check.cpp"),
         os.path.join(CSRC, "numerics.cpp"), "-o", exe],
        check=True, timeout=300)
    return exe


@pytest.mark.parametrize("ct,box,rcut,tol", [
    (0, (31.04, 31.04, 31.04), 9, 1e-5),
    (1, (52.0, 28.0, 70.0), 9, 1e-5),
    (1, (46.2, 46.2, 46.2), 9, 1e-6),
    (0, (142.0, 142.0, 142.0), 10, 1e-4)])
def test_plane_waves_from_the_tables(harm_check, ct, box, rcut, tol):
    r = subprocess.run([harm_check, str(ct), *map(str, box), str(rcut),
                        str(tol)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    m = re.search(r"failures 0 worst ([0-9.e+-]+)", r.stdout)
    assert m, r.stdout
    assert float(m.group(1)) < (1e-12 if ct else 3e-7 + 1e-12)


def test_no_plan_beyond_the_kernels(harm_check):
    """At tol 1e-7 the mixed path needs more degrees than its kernels hold."""
    r = subprocess.run([harm_check, "0", "46", "46", "46", "9", "1e-7"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "no plan" in r.stdout, r.stdout + r.stderr
