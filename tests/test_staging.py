"""Copies through the pinned slices (binarytpm_amd/csrc/staging.hip) on the CPU,
with host memory in the place of the device's: sizes around the limits, pinned
destinations, and memory that cannot be pinned, where the copy goes through the
runtime instead of failing."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "binarytpm_amd", "csrc")

PROGRAM = r"""
#include "staging.hip"
#include <cstdio>
#include <cstdlib>
static int fails = 0, copies = 0, fail_at = -1, mallocs = 0, live = 0, pinned = 0;
#define CHECK(c) do { if (!(c)) { std::printf("FAIL line %d: %s\n", __LINE__, #c); ++fails; } } while (0)
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (mallocs++ == fail_at) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  ++live;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); --live; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)&live; return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  ++copies;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  a->type = pinned ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return pinned == 2 ? hipErrorInvalidValue : hipSuccess;
}
}
std::string& btpm::last_error() { static std::string s; return s; }

// one copy each way of n bytes; returns how many the runtime made of it
static int run(btpm_ctx& c, size_t n, bool up) {
  std::vector<char> a(n), b(n, 0);
  for (size_t i = 0; i < n; i += 97) a[i] = (char)(i * 31 + 7);
  copies = 0;
  if (up) btpm::upload_staged(&c, b.data(), a.data(), n);
  else btpm::download_staged(&c, b.data(), a.data(), n);
  CHECK(a == b);
  return copies;
}

int main() {
  const size_t M = 1u << 20;
  btpm_ctx c;
  CHECK(run(c, 0, false) == 0 && run(c, 1, true) == 1);
  CHECK(run(c, 4 * M - 1, false) == 1 && run(c, 16 * M - 1, true) == 1);
  CHECK(mallocs == 0);
  // the first or the second slice cannot be pinned: one copy by the runtime,
  // nothing kept
  for (int k = 0; k < 2; ++k)
    for (int up = 0; up < 2; ++up) {
      mallocs = 0;
      fail_at = k;
      CHECK(run(c, 20 * M + 3, up) == 1);
      CHECK(live == 0 && c.stage[0] == nullptr && c.stage[1] == nullptr);
    }
  fail_at = -1;
  // and in slices again once it can
  CHECK(run(c, 4 * M, false) == 1 && run(c, 4 * M + 1, false) == 2 && run(c, 16 * M, true) == 4);
  CHECK(run(c, 20 * M + 3, false) == 4 && run(c, 130 * M + 1, true) == 5);
  CHECK(live == 2);
  pinned = 1;  // memory that HIP knows goes by one copy
  CHECK(run(c, 20 * M, false) == 1 && run(c, 20 * M, true) == 1);
  pinned = 2;  // what it cannot say anything about is pageable
  CHECK(run(c, 20 * M, false) == 4 && run(c, 20 * M, true) == 4);
  std::printf("%s\n", fails ? "FAILED" : "OK");
  return fails ? 1 : 0;
}
"""


def test_staged_copies(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    src = tmp_path / "staging.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "staging"
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc)))
    # host-only C++ on the definitions above in the place of the HIP runtime
    b = subprocess.run([os.path.join(rocm, "llvm", "bin", "clang++"), "-std=c++17", "-O1",
                        "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"), "-I", CSRC,
                        str(src), "-o", str(exe), "-lpthread"],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr
