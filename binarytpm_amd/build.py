"""Build libbtpm.so in-tree with hipcc for gfx950 (no JIT, no torch), and the
benchmark's calibration library libbtpm_probe.so (not part of the drop-in).

Usage: python -m binarytpm_amd.build   (or binarytpm_amd.build.build())
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SOURCES = ["conduct.hip", "linear_op.hip", "aux.hip", "stepwise.hip", "geometry.hip", "viewfactor.hip",
           "observe.hip", "io.hip", "staging.hip", "host.hip", "compat.hip", "noalloc.hip"]
LIB = os.path.join(HERE, "libbtpm.so")
PROBE_SRC = os.path.join(HERE, "bench_tools", "probe.hip")
PROBE_LIB = os.path.join(HERE, "libbtpm_probe.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # no packed FP32 (v_pk_*_f32) code generation: some of its forms have given
    # sporadic wrong results on this target, so every kernel is built without it
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _hipcc(srcs, out, verbose, extra=()):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    tmp = out + ".tmp"
    cmd = [hipcc, *HIPCC_FLAGS, "-I", CSRC, "-I", os.path.join(HERE, "..", "include"),
           *srcs, "-o", tmp, *extra]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"hipcc failed with status {res.returncode}")
    os.replace(tmp, out)


def build(verbose: bool = False) -> str:
    srcs = [os.path.join(CSRC, s) for s in SOURCES]
    _hipcc(srcs, LIB, verbose, ("-lpthread",))
    _hipcc([PROBE_SRC], PROBE_LIB, verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
