// fp32 values as sums of bf16 terms, for products on the bf16 matrix cores.
#pragma once

#include <hip/hip_runtime.h>

namespace wv {

// x as T terms, each rounding the remainder of the ones before it (to nearest
// even): two leave 2^-17 |x|, three 2^-25 |x|.
template <int T>
__device__ __forceinline__ void split_bf16(float x, __bf16 (&t)[T]) {
#pragma unroll
  for (int k = 0; k < T; ++k) {
    t[k] = (__bf16)x;
    x -= (float)t[k];
  }
}

// The same of every element of a vector.
template <int T, class F, class B>
__device__ __forceinline__ void split_bf16(F x, B (&t)[T]) {
#pragma unroll
  for (int k = 0; k < T; ++k)
#pragma unroll
    for (int e = 0; e < (int)(sizeof(B) / sizeof(__bf16)); ++e) {
      t[k][e] = (__bf16)x[e];
      x[e] -= (float)t[k][e];
    }
}

}  // namespace wv
