// mla_values.hpp -- values of stored MLA rows and staged queries, as the
// single-query kernel and the batched path's kernels read them.
#pragma once

#include "grm_common.hpp"

namespace grm {
namespace mla {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// q[0, N) in order through `use(value, index)`, read from LDS kAhead values
// ahead of their use: a lone wave on its SIMD would otherwise wait for LDS
// (over 100 cycles) at every chunk of its serial fp64 chain.
template <int N, int kAhead, typename F>
__device__ __forceinline__ void stream_lds(const double* __restrict__ q, F use) {
  static_assert(N % kAhead == 0, "whole stages");
  double cur[kAhead], nxt[kAhead];
#pragma unroll
  for (int e = 0; e < kAhead; ++e) cur[e] = q[e];
#pragma unroll
  for (int s = 0; s < N / kAhead; ++s) {
    if (s + 1 < N / kAhead) {
#pragma unroll
      for (int e = 0; e < kAhead; ++e) nxt[e] = q[(s + 1) * kAhead + e];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int e = 0; e < kAhead; ++e) use(cur[e], s * kAhead + e);
#pragma unroll
    for (int e = 0; e < kAhead; ++e) cur[e] = nxt[e];
  }
}

// Value i of a chunk (fp32 or bf16) as a double.
template <int DT>
__device__ __forceinline__ double chunk_value(u32x4 v, int i) {
  const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
  if constexpr (DT == kF32) {
    return static_cast<double>(__uint_as_float(w4[i]));
  } else {
    const uint32_t w = w4[i >> 1];
    return static_cast<double>(__uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16)));
  }
}

// The law's query norm from the staged query (zeros past dim add nothing):
// one serial fp64 chain over d (cpp/grm_runtime.cpp:4310-4314).  n is a
// multiple of 4.
__device__ inline double staged_norm(const double* __restrict__ qd, uint32_t n) {
  double acc = 0.0;
  uint32_t d = 0;
  for (; d + 64 <= n; d += 64) stream_lds<64, 16>(qd + d, [&](double q, int) { acc = fma(q, q, acc); });
  for (; d < n; d += 4) stream_lds<4, 4>(qd + d, [&](double q, int) { acc = fma(q, q, acc); });
  return sqrt(acc);
}

}  // namespace mla
}  // namespace grm
