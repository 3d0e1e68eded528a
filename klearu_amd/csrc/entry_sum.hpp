// entry_sum.hpp -- a neuron's sequential sum over an input's nonzeros (neuron.rs:47-62),
// the weights of the next kEntries entries in flight while the ones before are added.
#pragma once
#include "common.hpp"

namespace kh {

constexpr int kEntries = 16;
__host__ __device__ constexpr int entries_padded(int nnz) {
  return (nnz + 2 * kEntries - 1) / (2 * kEntries) * (2 * kEntries);
}

// sum_e weight(nzi[e]) * nzv[e] in order, from -0.0, for nnz > 0.  The lists are in LDS
// (four entries a read) and padded to entries_padded(nnz) with entries that may be
// loaded; in the last, partial group their products are replaced by -0.0, which
// leaves a sum as it is.
template <typename W>
__device__ __forceinline__ float sum_entries(const uint32_t* nzi, const float* nzv, int nnz, W&& weight) {
  const int npad = entries_padded(nnz);
  float s = -0.0f, w0[kEntries], w1[kEntries];
  auto load = [&](float (&w)[kEntries], int e0) {
#pragma unroll
    for (int u = 0; u < kEntries; ++u) w[u] = weight(nzi[e0 + u]);
  };
  auto add = [&](const float (&w)[kEntries], int e0) {
#pragma unroll
    for (int u = 0; u < kEntries; ++u) s = __fadd_rn(s, __fmul_rn(w[u], nzv[e0 + u]));
    asm volatile("" : "+v"(s));   // these sums stay ahead of the next loads
  };
  auto add_some = [&](const float (&w)[kEntries], int e0) {
#pragma unroll
    for (int u = 0; u < kEntries; ++u) {
      const float p = __fmul_rn(w[u], nzv[e0 + u]);
      s = __fadd_rn(s, e0 + u < nnz ? p : -0.0f);
    }
  };
  load(w0, 0);
  int e0 = 0;
  for (; e0 + 2 * kEntries <= nnz; e0 += 2 * kEntries) {
    load(w1, e0 + kEntries);
    add(w0, e0);
    load(w0, min(e0 + 2 * kEntries, npad - kEntries));
    add(w1, e0 + kEntries);
  }
  if (e0 < nnz) {
    load(w1, e0 + kEntries);
    add_some(w0, e0);
    add_some(w1, e0 + kEntries);
  }
  return s;
}

// Whether offsets into a transposed copy [dim][n] fit 32 bits in bytes: the lists then
// hold d * n, and a weight's address is one 32-bit add (five vector instructions per
// entry instead of some twenty with 64-bit scalar products, which bounded the kernel).
__host__ __device__ constexpr bool offsets_fit(int64_t dim, int64_t n) { return dim * n < ((int64_t)1 << 30); }
__device__ __forceinline__ float weight_at(const float* __restrict__ W, uint32_t i) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(W) + (i << 2));
}

}  // namespace kh
