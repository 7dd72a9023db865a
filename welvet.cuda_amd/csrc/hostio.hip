// Copies between pinned host memory and device memory by a kernel.
#include "kernels.h"

namespace wv {
namespace {

// Two ranges in one launch: the first `blocks0` workgroups copy the first.
// 16-byte accesses over whole vectors, then the 4-byte words left over. Bound
// by the host link, and below about 256 KB by its latency (one load in flight
// per lane is enough: 256 workgroups keep 1 MiB in flight).
constexpr int kThreads = 256;

__device__ __forceinline__ void copy_range(const CopyRange& r, int block, int blocks) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const size_t vecs = r.bytes / 16, step = (size_t)blocks * kThreads;
  const size_t first = (size_t)block * kThreads + threadIdx.x;
  const f32x4* src = static_cast<const f32x4*>(r.src);
  f32x4* dst = static_cast<f32x4*>(r.dst);
  for (size_t i = first; i < vecs; i += step) dst[i] = src[i];
  const size_t words = r.bytes / 4;
  for (size_t i = 4 * vecs + first; i < words; i += step)
    static_cast<uint32_t*>(r.dst)[i] = static_cast<const uint32_t*>(r.src)[i];
}

__global__ __launch_bounds__(kThreads) void k_copy(CopyRange a, CopyRange b, int blocks_a) {
  if ((int)blockIdx.x < blocks_a) copy_range(a, blockIdx.x, blocks_a);
  else copy_range(b, blockIdx.x - blocks_a, gridDim.x - blocks_a);
}

int blocks_of(size_t bytes) {
  const size_t n = (bytes + 16 * kThreads - 1) / (16 * kThreads);
  return n < 128 ? (int)n : 128;
}

}  // namespace

Status launch_copy(const CopyRange& a, const CopyRange& b, hipStream_t st) {
  for (const CopyRange* r : {&a, &b})
    if (r->bytes && (!r->dst || !r->src || r->bytes % 4 != 0 ||
                     ((reinterpret_cast<uintptr_t>(r->dst) | reinterpret_cast<uintptr_t>(r->src)) & 15)))
      return Status::err(kInvalid, "copy: 16-byte aligned buffers of whole words");
  const int na = blocks_of(a.bytes), nb = blocks_of(b.bytes);
  if (na + nb == 0) return Status::ok();
  k_copy<<<na + nb, kThreads, 0, st>>>(a, b, na);
  return hip_status(hipGetLastError(), "copy launch");
}

}  // namespace wv
