// staging.hip -- copies between the device and pageable host memory through a
// context's two pinned slices (host code).
#include <hip/hip_runtime.h>

#include <cstring>
#include <system_error>
#include <thread>

#include "runtime.h"

namespace btpm {
namespace {
// Copies between the device and pageable memory, in slices through two pinned
// buffers.  Measured on 64 MB: to a host buffer of untouched 4 KB pages the
// runtime's own copy reaches 3.9 GB/s (untouched 2 MB pages 10.8, a touched
// buffer 7 to 18), since it takes the page faults on one thread; eight threads
// behind the DMA reach 33 to 40.  From 4 MB on the staged copy is the faster
// one down, and from 16 MB on up (64 MB: 37 GB/s against 47), where there is
// nothing to fault in.  A quarter of the copy per slice keeps DMA and threads
// both busy; slices of 2 MB lose the gain to starting the threads.
constexpr size_t kStageSlice = 32u << 20, kStageSliceMin = 4u << 20;
constexpr size_t kStageDown = 4u << 20, kStageUp = 16u << 20;

size_t stage_slice(size_t bytes) {
  const size_t quarter = ((bytes + 3) / 4 + 4095) & ~(size_t)4095;
  return std::min(kStageSlice, std::max(kStageSliceMin, quarter));
}

// memory that HIP knows (pinned, managed, device) goes by DMA alone
bool dma_ready(const void* p) {
  hipPointerAttribute_t a = {};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// False where memory cannot be pinned: the runtime's own copy does without.
// (Two slices take 0.8 ms to pin, as much as the runtime's copy of 4 MB.)
bool stage_buffers(btpm_ctx* ctx) {
  for (int k = 0; k < 2; ++k)
    if (!ctx->stage_ev[k])
      HIPCHK(hipEventCreateWithFlags(&ctx->stage_ev[k], hipEventDisableTiming));
  if (ctx->stage[0]) return true;
  char* p[2] = {nullptr, nullptr};
  for (int k = 0; k < 2; ++k)
    if (hipHostMalloc((void**)&p[k], kStageSlice, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      if (k) (void)hipHostFree(p[0]);
      return false;
    }
  ctx->stage[0] = p[0];
  ctx->stage[1] = p[1];
  return true;
}

// memcpy split over up to 8 host threads (pageable <-> pinned slices)
void par_memcpy(char* d, const char* s, size_t n) {
  const int nt = (int)std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
  const size_t part = (n + nt - 1) / nt;
  std::vector<std::thread> pool;
  pool.reserve(nt);  // nothing to throw between a thread's start and its join
  for (int t = 1; t < nt; ++t) {
    const size_t a = std::min(n, (size_t)t * part), b = std::min(n, a + part);
    if (a >= b) continue;
    try {
      pool.emplace_back([=] { std::memcpy(d + a, s + a, b - a); });
    } catch (const std::system_error&) {
      std::memcpy(d + a, s + a, b - a);  // no thread to spare: copy here
    }
  }
  std::memcpy(d, s, std::min(n, part));
  for (auto& th : pool) th.join();
}
}  // namespace

void upload_staged(btpm_ctx* ctx, void* dst, const void* src, size_t bytes) {
  hipStream_t st = ctx->stream;
  if (bytes < kStageUp || dma_ready(src) || !stage_buffers(ctx)) {
    if (bytes) HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st));
    return;
  }
  const char* s = static_cast<const char*>(src);
  char* d = static_cast<char*>(dst);
  const size_t slice = stage_slice(bytes);
  size_t i = 0;
  for (size_t off = 0; off < bytes; off += slice, ++i) {
    const size_t n = std::min(slice, bytes - off);
    const int k = (int)(i & 1);
    // this buffer's previous slice has left for the device
    if (i >= 2) HIPCHK(hipEventSynchronize(ctx->stage_ev[k]));
    par_memcpy(ctx->stage[k], s + off, n);
    HIPCHK(hipMemcpyAsync(d + off, ctx->stage[k], n, hipMemcpyHostToDevice, st));
    HIPCHK(hipEventRecord(ctx->stage_ev[k], st));
  }
  HIPCHK(hipStreamSynchronize(st));
}

void download_staged(btpm_ctx* ctx, void* dst, const void* src, size_t bytes) {
  hipStream_t st = ctx->stream;
  if (bytes < kStageDown || dma_ready(dst) || !stage_buffers(ctx)) {
    if (bytes) HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return;
  }
  const char* s = static_cast<const char*>(src);
  char* d = static_cast<char*>(dst);
  const size_t slice = stage_slice(bytes), ns = (bytes + slice - 1) / slice;
  auto issue = [&](size_t j) {
    const size_t off = j * slice, n = std::min(slice, bytes - off);
    HIPCHK(hipMemcpyAsync(ctx->stage[j & 1], s + off, n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipEventRecord(ctx->stage_ev[j & 1], st));
  };
  issue(0);
  for (size_t j = 0; j < ns; ++j) {
    // the other buffer's slice was copied out in the previous pass
    if (j + 1 < ns) issue(j + 1);
    HIPCHK(hipEventSynchronize(ctx->stage_ev[j & 1]));
    const size_t off = j * slice;
    par_memcpy(d + off, ctx->stage[j & 1], std::min(slice, bytes - off));
  }
}
}  // namespace btpm
