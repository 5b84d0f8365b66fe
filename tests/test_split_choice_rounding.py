"""The two launches of a call without host positions decide, each on the device,
which of them images the job (split_wins, csrc/sarbp_poly.h).  Contracted to
FMAs in one and not in the other, its sums would round differently and a job at
the limit would be imaged twice or not at all: compiled for the device it holds
no FP64 FMA."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sar_cambrianaccelerationcard_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

SOURCE = """
#include <hip/hip_runtime.h>
#include "sarbp_poly.h"
__global__ void choice(sarbp::BpArgs a, int rows, int* out) {
  *out = sarbp::split_wins(a, a.pos, rows, a.split_limit);
}
"""


def test_choice_is_not_contracted(tmp_path):
    src, asm = str(tmp_path / "choice.hip"), str(tmp_path / "choice.s")
    with open(src, "w") as f:
        f.write(SOURCE)
    b = subprocess.run([os.path.join(ROCM, "bin", "hipcc"), "--offload-arch=gfx950", "--cuda-device-only", "-S", "-O3",
                        "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        f"-I{ROOT}/include", f"-I{CSRC}", src, "-o", asm],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    with open(asm) as f:
        text = f.read()
    assert "v_mul_f64" in text and "v_add_f64" in text
    assert "_fma_f64" not in text and "_fmac_f64" not in text
