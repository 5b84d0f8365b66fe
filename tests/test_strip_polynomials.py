"""The row-polynomial setup of the BP kernels (csrc/sarbp_poly.h) on the CPU:
tests/host/strip_poly_check.cpp compiles the header that the kernels compile and
checks its windows and bounds against the exact slant range."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sar_cambrianaccelerationcard_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("strip_poly") / "strip_poly_check")
    # no contraction: the FP32 results are those of the kernels' code
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                        f"-I{ROOT}/include", f"-I{CSRC}", os.path.join(CSRC, "sarbp_plan.cpp"),
                        os.path.join(ROOT, "tests", "host", "strip_poly_check.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    return exe


@pytest.mark.parametrize("check", ["window", "ref", "df", "df_phase", "bins", "root", "split", "launch"])
def test_strip_polynomials(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=300)
    print(r.stdout, r.stderr[-4000:])
    assert r.returncode == 0, r.stdout + r.stderr[-4000:]
