"""Launch widths of the operator's kernels (binarytpm_amd/csrc/runtime.h) follow
the device's compute units, on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "binarytpm_amd", "csrc")

PROGRAM = r"""
#include "runtime.h"
using namespace btpm;
int main() {
  int bad = 0;
  for (int cus : {32, 64, 256}) {
    bad += smooth_lin_width(1, cus) != 16 || smooth_lin_width(80LL * cus, cus) != 16;
    bad += smooth_lin_width(80LL * cus + 1, cus) != 32 || smooth_lin_width(1LL << 40, cus) != 32;
    bad += crater_lin_width(1, cus) != 2 || crater_lin_width(2LL * cus, cus) != 2;
    bad += crater_lin_width(2LL * cus + 1, cus) != 5 || crater_lin_width(1LL << 40, cus) != 5;
  }
  return bad;
}
"""


def test_widths(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(PROGRAM)
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")
    b = subprocess.run([hipcc, "-x", "c++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                        "-I", include, "-I", CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-2000:]
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
