// chain_add.hpp -- sequential f32 sums over terms that other waves put in LDS.
#pragma once

#include "common.hpp"

namespace kh {

// Sequential sums r + t[0] + t[1] + ... over quads of one chain's terms in LDS
// (quad q of this lane's chain at base[q * C]), with the LDS reads of the next
// eight quads issued before the adds of the current ones and pinned there
// (left to the scheduler, each read sinks to its first use and the chain waits
// out the LDS latency every four adds).
__device__ __forceinline__ float add_quads8(const float4* v, float r) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    r = r + v[b].x;
    r = r + v[b].y;
    r = r + v[b].z;
    r = r + v[b].w;
  }
  return r;
}

// NQ (a multiple of 8) quads, fully unrolled: every register index is a
// compile-time constant, so no value is copied.
template <int NQ, int C>
__device__ __forceinline__ float chain_add_static(const float4* base, float r) {
  static_assert(NQ % 8 == 0, "whole groups of quads");
  float4 v[16];
#pragma unroll
  for (int b = 0; b < 8; ++b) v[b] = base[b * C];
#pragma unroll
  for (int g = 0; g < NQ / 8; ++g) {
    if (g + 1 < NQ / 8) {
#pragma unroll
      for (int b = 0; b < 8; ++b) v[((g + 1) % 2) * 8 + b] = base[((g + 1) * 8 + b) * C];
    }
    __builtin_amdgcn_sched_barrier(0);
    r = add_quads8(&v[(g % 2) * 8], r);
  }
  return r;
}

}  // namespace kh
