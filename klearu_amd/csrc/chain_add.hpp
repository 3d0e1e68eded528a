// chain_add.hpp -- sequential f32 sums over terms that other waves put in LDS.
#pragma once

#include "common.hpp"

namespace kh {

// Sequential sums r + t[0] + t[1] + ... over quads of one chain's terms in LDS
// (quad q of this lane's chain at base[q * C]), with the LDS reads of the next
// group of quads issued before the adds of the current one and pinned there (left
// to the scheduler, each read sinks to its first use and the chain waits out the
// LDS latency every four adds).
template <int N>
__device__ __forceinline__ float add_quads(const float4* v, float r) {
#pragma unroll
  for (int b = 0; b < N; ++b) {
    r = r + v[b].x;
    r = r + v[b].y;
    r = r + v[b].z;
    r = r + v[b].w;
  }
  // keeps the adds here: free of side effects, they would sink below the reads of
  // all later groups, whose values then take hundreds of registers
  asm volatile("" : "+v"(r));
  return r;
}

// NQ quads (whole groups of kChainGroup, or fewer), fully unrolled: every register
// index is a compile-time constant, so no value is copied.
constexpr int kChainGroup = 16;
template <int NQ, int C>
__device__ __forceinline__ float chain_add_static(const float4* base, float r) {
  constexpr int G = NQ < kChainGroup ? NQ : kChainGroup;
  static_assert(NQ % G == 0, "whole groups of quads");
  float4 v[2 * G];
#pragma unroll
  for (int b = 0; b < G; ++b) v[b] = base[b * C];
#pragma unroll
  for (int g = 0; g < NQ / G; ++g) {
    if (g + 1 < NQ / G) {
#pragma unroll
      for (int b = 0; b < G; ++b) v[((g + 1) % 2) * G + b] = base[((g + 1) * G + b) * C];
    }
    __builtin_amdgcn_sched_barrier(0);
    r = add_quads<G>(&v[(g % 2) * G], r);
  }
  return r;
}

// Products of up to 64 chains in LDS, two chunks of STEP steps: quad q (steps
// 4q..4q+3) of chain c at q[chunk & 1][q * kStride + c].
constexpr int kChainAhead = 4;  // chunks in flight per producer thread (default)
template <int STEP, int CHAINS>
struct ChainLds {
  static constexpr int kStep = STEP, kChains = CHAINS;
  static constexpr int kStride = CHAINS == 1 ? 1 : CHAINS + 1;
  float4 q[2][STEP / 4 * kStride];
};

// The block steps through nch chunks: waves 1.. (producers) put chunk c's
// products into LDS buffer c & 1 with make(c, u) (u = c % AHEAD, the
// thread's register slot) and there request chunk c + AHEAD; wave 0 adds
// the chunk before, lane l chain l, and returns s0 + every term in order.  A wave
// with `idle` set (the whole wave) only keeps the barriers.  The
// loop has no branch around a load (chunks past the end are clamped, formed and
// not added): behind a branch the compiler waits for every load in flight.
template <int AHEAD = kChainAhead, typename Lds, typename Make>
__device__ __forceinline__ float chain_run(Lds& lds, int nch, float s0, Make make, bool idle = false) {
  const int lane = threadIdx.x & 63;
  float s = s0;
  if (idle) {
    const int last = (nch + AHEAD - 1) / AHEAD * AHEAD;
    for (int c = 0; c < last; ++c) lds_barrier();
  } else if (threadIdx.x >= 64) {
    for (int c0 = 0; c0 < nch; c0 += AHEAD) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        make(c0 + u, u);
        lds_barrier();
        // left alone, the scheduler forms every slot's products before the first
        // barrier, and so waits for the last slot's loads there
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    const int last = (nch + AHEAD - 1) / AHEAD * AHEAD;
    for (int c = 0; c < last; ++c) {
      lds_barrier();
      if (c < nch) {
        const float4* q = &lds.q[c & 1][min(lane, Lds::kChains - 1)];
        s = chain_add_static<Lds::kStep / 4, Lds::kStride>(q, s);
      }
    }
  }
  return s;
}

}  // namespace kh
