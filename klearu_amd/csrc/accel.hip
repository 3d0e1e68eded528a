// accel.hip -- klearu-accel entry points on the GPU (gfx950).
//
// Replaces dense_dot_dense_simd / sparse_dot_dense_simd / scatter_add_simd
// (crates/klearu-accel/src/simd/mod.rs:19-109) and the Bf16Weights /
// Bf16FullMode methods (crates/klearu-accel/src/bf16/mod.rs:37-134).
//
// The reference's x86_64 kernels fix a summation order (simd/mod.rs:145-236):
// 16 (dense) or 8 (sparse) FMA lanes over chunks, a fixed horizontal-add tree,
// then a scalar tail.  Here each of those accumulator lanes is a GPU lane
// running the same FMA chain, so the results are bit-identical.  The BF16
// dots are sequential sums and run as one chain per row.
#include "chain_add.hpp"

namespace kh {

// ((v0+v4)+(v1+v5)) + ((v2+v6)+(v3+v7)), the hsum_avx2 tree (simd/mod.rs:128-141).
__device__ __forceinline__ float hsum8_tree(const float v[8]) {
  const float s0 = v[0] + v[4], s1 = v[1] + v[5], s2 = v[2] + v[6], s3 = v[3] + v[7];
  return (s0 + s1) + (s2 + s3);
}

// One 16-lane group per row; 4 rows per wave.  A lane's chain is n / 16 FMAs, so
// what counts is the rows' bytes in flight: kDdAhead chunks are requested while
// the kDdAhead before them are added.  11008 x 4096 (180 MB): 33 us, 5.4 TB/s
// (85 us with one chunk at a time).
constexpr int kDdAhead = 16;
__global__ __launch_bounds__(256) void dense_dot_kernel(const float* __restrict__ a, int64_t rows,
                                                        int64_t lda, const float* __restrict__ b,
                                                        int64_t n, float* __restrict__ out) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t row = gid >> 4;
  const int l = threadIdx.x & 15;
  const bool ok = row < rows;
  const float* __restrict__ ar = a + (ok ? row : 0) * lda;
  const int64_t chunks = n / 16, full = chunks / kDdAhead * kDdAhead;
  float acc = 0.0f;
  float a0[kDdAhead], a1[kDdAhead], b0[kDdAhead], b1[kDdAhead];
  // the last group's request past the end repeats the group before it
  auto load = [&](float (&av)[kDdAhead], float (&bv)[kDdAhead], int64_t c) {
    const int64_t c1 = min(c, full - kDdAhead);
#pragma unroll
    for (int u = 0; u < kDdAhead; ++u) av[u] = ar[(c1 + u) * 16 + l];
#pragma unroll
    for (int u = 0; u < kDdAhead; ++u) bv[u] = b[(c1 + u) * 16 + l];
  };
  auto add = [&](const float (&av)[kDdAhead], const float (&bv)[kDdAhead]) {
#pragma unroll
    for (int u = 0; u < kDdAhead; ++u) acc = fmaf(av[u], bv[u], acc);
  };
  int64_t c = 0;
  if (full > 0) {
    load(a0, b0, 0);
    for (; c + kDdAhead < full; c += 2 * kDdAhead) {
      load(a1, b1, c + kDdAhead);
      __builtin_amdgcn_sched_barrier(0);
      add(a0, b0);
      load(a0, b0, c + 2 * kDdAhead);
      __builtin_amdgcn_sched_barrier(0);
      add(a1, b1);
    }
    if (c < full) add(a0, b0);
  }
  for (c = full; c < chunks; ++c) acc = fmaf(ar[c * 16 + l], b[c * 16 + l], acc);
  const int64_t rs = chunks * 16;
  const bool extra = rs + 8 <= n;
  if (extra && l < 8) acc = fmaf(ar[rs + l], b[rs + l], acc);
  // lane l < 8 holds acc0[l], lane l+8 holds acc1[l]
  const float other = __shfl_down(acc, 8, 16);
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = __shfl(acc + other, i, 16);
  if (!ok || l != 0) return;
  float sum = hsum8_tree(v);
  for (int64_t i = extra ? rs + 8 : rs; i < n; ++i) sum = __fadd_rn(sum, __fmul_rn(ar[i], b[i]));
  out[row] = sum;
}

// The whole block gathers a tile of (value, dense value) pairs into LDS, then
// lanes 0..7 run the reference's eight FMA lanes over it, so a call waits for two
// dependent loads per tile and not per 8 entries (75 entries: 8.1 -> 4.9 us).
constexpr int kSdTile = 2048;
__global__ __launch_bounds__(256) void sparse_dot_kernel(const uint32_t* __restrict__ idx,
                                                         const float* __restrict__ val, int64_t nnz,
                                                         const float* __restrict__ dense,
                                                         float* __restrict__ out) {
  __shared__ float sv[kSdTile], sd[kSdTile];
  constexpr int kPer = kSdTile / 256;
  const int l = threadIdx.x;
  const int64_t chunks = nnz / 8;
  float acc = 0.0f, sum = 0.0f;
  for (int64_t e0 = 0; e0 < nnz; e0 += kSdTile) {
    uint32_t id[kPer];
    float v[kPer], d[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int64_t e = min(e0 + u * 256 + l, nnz - 1);
      id[u] = idx[e];
      v[u] = val[e];
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) d[u] = dense[id[u]];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      sv[u * 256 + l] = v[u];
      sd[u * 256 + l] = d[u];
    }
    __syncthreads();
    const int64_t left = chunks * 8 - e0;
    const int m = (int)(left < 0 ? 0 : left < kSdTile ? left : kSdTile);
    if (l < 8)
      for (int e = l; e < m; e += 8) acc = fmaf(sv[e], sd[e], acc);
    if (e0 + kSdTile >= nnz && l < 64) {   // last tile: the lanes' sum, then the scalar tail
      float t[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) t[i] = __shfl(acc, i, 64);
      sum = hsum8_tree(t);
      const int end = (int)(nnz - e0);
      for (int e = m; e < end; ++e) sum = __fadd_rn(sum, __fmul_rn(sv[e], sd[e]));
    }
  }
  if (l == 0) *out = sum;
}

// Deterministic scatter-add: chunks of 1024 entries in order; within a chunk the
// first occurrence of each index applies all of that index's updates in entry
// order, one rounded add at a time (as scatter_add_avx2's scalar stores).  An LDS
// hash table of entry positions finds each index's first entry and its count, so
// only an index that repeats looks through the chunk (75 entries: 11.6 -> 4.5 us
// against a look through all earlier and later entries by every thread).
constexpr int kSaSlots = 2048;
__global__ __launch_bounds__(1024) void scatter_add_kernel(const uint32_t* __restrict__ idx,
                                                           const float* __restrict__ val,
                                                           int64_t n, float* __restrict__ dense,
                                                           float scale) {
  __shared__ uint32_t sidx[1024];
  __shared__ float sval[1024];
  __shared__ int rep[kSaSlots];    // 1 + position of an entry with the slot's index; 0: free
  __shared__ int first[kSaSlots], count[kSaSlots];
  const int t = threadIdx.x;
  for (int64_t c0 = 0; c0 < n; c0 += 1024) {
    const int m = (int)min<int64_t>(1024, n - c0);
    const uint32_t me = idx[c0 + min(t, m - 1)];
    const float v = __fmul_rn(val[c0 + min(t, m - 1)], scale);
    sidx[t] = me;
    sval[t] = v;
    for (int s = t; s < kSaSlots; s += 1024) {
      rep[s] = 0;
      first[s] = 1024;
      count[s] = 0;
    }
    const float d0 = dense[me];   // no entry of this chunk is applied before the next barrier
    __syncthreads();
    int slot = 0;
    if (t < m) {
      slot = (int)((me * 2654435761u) >> 21);
      for (;;) {   // at most 1024 indices in 2048 slots: a free or matching slot comes
        const int r = atomicCAS(&rep[slot], 0, t + 1);
        if (r == 0 || sidx[r - 1] == me) break;
        slot = (slot + 1) & (kSaSlots - 1);
      }
      atomicMin(&first[slot], t);
      atomicAdd(&count[slot], 1);
    }
    __syncthreads();
    if (t < m && first[slot] == t) {
      float d = __fadd_rn(d0, v);
      int more = count[slot] - 1;
      for (int j = t + 1; more > 0; ++j)
        if (sidx[j] == me) {
          d = __fadd_rn(d, sval[j]);
          --more;
        }
      dense[me] = d;
    }
    __syncthreads();
  }
}

// Elementwise kernels: eight elements per access (16 bytes of BF16, 32 of f32) and
// kEwGroups of them in flight per thread where both arrays are 16-byte aligned;
// one element per thread otherwise; the last block also takes the last n % 8 (in a launch of
// their own they cost a call 2.6 us).  45 M elements, BF16
// from f32 / f32 from BF16 (271 MB): 57 / 48 us, against 98 / 93 us with one
// element per thread.
constexpr int kEwGroups = 4;
constexpr int kEwBlock = 256 * kEwGroups * 8;   // elements per block

struct EwFromF32 {
  using In = float;
  using Out = uint16_t;
  static __device__ __forceinline__ uint16_t at(float x, uint16_t) { return f32_to_bf16(x); }
  static constexpr bool kReadOut = false;
};
struct EwToF32 {
  using In = uint16_t;
  using Out = float;
  static __device__ __forceinline__ float at(uint16_t x, float) { return bf16_to_f32(x); }
  static constexpr bool kReadOut = false;
};
struct EwUpdate {
  using In = float;
  using Out = uint16_t;
  static __device__ __forceinline__ uint16_t at(float d, uint16_t w) {
    return f32_to_bf16(__fadd_rn(bf16_to_f32(w), d));
  }
  static constexpr bool kReadOut = true;
};

template <typename T>
struct alignas(16) EwVec {
  T v[8];
};

template <typename Op>
__global__ __launch_bounds__(256) void ew_vec_kernel(const typename Op::In* __restrict__ x,
                                                     typename Op::Out* __restrict__ o, int64_t n) {
  using VI = EwVec<typename Op::In>;
  using VO = EwVec<typename Op::Out>;
  const int64_t n8 = n / 8;
  const int64_t g0 = (int64_t)blockIdx.x * 256 * kEwGroups + threadIdx.x;
  const VI* __restrict__ xv = reinterpret_cast<const VI*>(x);
  VO* __restrict__ ov = reinterpret_cast<VO*>(o);
  VI a[kEwGroups];
  VO r[kEwGroups];
#pragma unroll
  for (int u = 0; u < kEwGroups; ++u) {
    const int64_t g = min(g0 + u * 256, n8 - 1);
    a[u] = xv[g];
    if (Op::kReadOut) r[u] = ov[g];
  }
#pragma unroll
  for (int u = 0; u < kEwGroups; ++u) {
    const int64_t g = g0 + u * 256;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[u].v[i] = Op::at(a[u].v[i], r[u].v[i]);
    if (g < n8) ov[g] = r[u];
  }
  const int64_t i = n8 * 8 + threadIdx.x;
  if (blockIdx.x + 1 == gridDim.x && i < n) o[i] = Op::at(x[i], o[i]);
}

template <typename Op>
__global__ __launch_bounds__(256) void ew_kernel(const typename Op::In* __restrict__ x,
                                                 typename Op::Out* __restrict__ o, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) o[i] = Op::at(x[i], o[i]);
}

template <typename Op>
static int ew_launch(const typename Op::In* x, typename Op::Out* o, int64_t n, hipStream_t st) {
  if (n == 0) return KH_OK;
  if (n >= 8 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(o)) & 15) == 0)
    hipLaunchKernelGGL(ew_vec_kernel<Op>, dim3((unsigned)ceil_div(n, kEwBlock)), dim3(256), 0, st, x, o, n);
  else
    hipLaunchKernelGGL(ew_kernel<Op>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, st, x, o, n);
  KH_LAUNCHED();
  return KH_OK;
}

// Sequential sums of rows (Bf16Weights::dot_f32's iterator sum from -0.0): a chain
// of n dependent adds per row bounds a call, so producer waves form the products
// in LDS, kChainAhead chunks of weights in flight, and wave 0 adds, four per read.
// ROWS rows per block: 16 when there are several, 1 (and longer chunks) for one.
// One row of 4096: 12.2 us (about 9 us of adds), against 316 us with one lane
// loading and adding.
template <int ROWS>
struct BdShape {
  static constexpr int kStep = ROWS == 1 ? 512 : 128;
  static constexpr int kProd = kStep / 4 * ROWS;
  static constexpr int kThreads = 64 + kProd;
};

__device__ __forceinline__ float bd_f32(float x) { return x; }
__device__ __forceinline__ float bd_f32(uint16_t x) { return bf16_to_f32(x); }
template <typename T>
struct alignas(4 * sizeof(T)) BdQuad {
  T v[4];
};
// Elements k..k+3 of p (past n: the last one).  VEC: one access, n a multiple of 4
// and p aligned to four elements.
template <bool VEC, typename T>
__device__ __forceinline__ BdQuad<T> bd_load(const T* __restrict__ p, int64_t k, int64_t n) {
  if constexpr (VEC) return *reinterpret_cast<const BdQuad<T>*>(p + min(k, n - 4));
  BdQuad<T> q;
#pragma unroll
  for (int i = 0; i < 4; ++i) q.v[i] = p[min(k + i, n - 1)];
  return q;
}

template <int ROWS, bool VEC, typename TX>
__global__ __launch_bounds__(BdShape<ROWS>::kThreads) void bf16_dot_kernel(
    const uint16_t* __restrict__ w, int64_t rows, int64_t ldw, const TX* __restrict__ x, int64_t n,
    float* __restrict__ o) {
  constexpr int kStep = BdShape<ROWS>::kStep;
  using Lds = ChainLds<kStep, ROWS>;
  __shared__ Lds lds;
  const int pt = (int)threadIdx.x - 64;
  const int i = pt & (ROWS - 1), k4 = pt / ROWS;
  const int64_t r0 = (int64_t)blockIdx.x * ROWS;
  const uint16_t* __restrict__ wr = w + min(r0 + i, rows - 1) * ldw;
  const int nch = (int)((n + kStep - 1) / kStep);
  BdQuad<uint16_t> wv[kChainAhead];
  BdQuad<TX> xv[kChainAhead];
  auto fetch = [&](int64_t c, int u) {
    const int64_t k = c * kStep + 4 * k4;
    wv[u] = bd_load<VEC>(wr, k, n);
    xv[u] = bd_load<VEC>(x, k, n);
  };
  if (pt >= 0 && nch > 0) {
#pragma unroll
    for (int u = 0; u < kChainAhead; ++u) fetch(u, u);
  }
  const float s = chain_run(lds, nch, -0.0f, [&](int c, int u) {
    const int64_t k = (int64_t)c * kStep + 4 * k4;
    float p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = k + q < n ? __fmul_rn(bf16_to_f32(wv[u].v[q]), bd_f32(xv[u].v[q])) : -0.0f;
    lds.q[c & 1][k4 * Lds::kStride + i] = make_float4(p[0], p[1], p[2], p[3]);
    fetch(c + kChainAhead, u);
  });
  if (threadIdx.x < ROWS && r0 + (int)threadIdx.x < rows) o[r0 + threadIdx.x] = s;
}

// The same sums with a row per thread: no chain is fed, but a block of 576 threads for 16
// rows costs about 0.45 us a thousand rows before it adds anything.  This form takes 2 us
// and 0.09 us per element of a row until the chip is full, hence bd_short: us for 32000 rows,
// rows per thread / chains, 16 elements 2.5 / 16.5, 160 elements 16.1 / 20.7, 256 elements
// 24.2 / 23.4; 2000 rows of 16 3.3 / 3.5, of 32 4.6 / 3.7.  A lane reads its row alone, so
// past the L2 (32 MB) a row's lines come more than once: 64000 rows of 256 35.7 / 45.6,
// 128000 of 128 60.7 / 85.2, of 160 84.1 / 78.9.
template <typename TX>
__global__ __launch_bounds__(64) void bf16_dot_rows_kernel(const uint16_t* __restrict__ w, int64_t rows, int64_t ldw,
                                                           const TX* __restrict__ x, int64_t n, float* __restrict__ o) {
  const int64_t r = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (r >= rows) return;
  const uint16_t* __restrict__ wr = w + r * ldw;
  float s = -0.0f;
  for (int64_t i = 0; i < n; ++i) s = __fadd_rn(s, __fmul_rn(bf16_to_f32(wr[i]), bd_f32(x[i])));
  o[r] = s;
}
static bool bd_short(int64_t rows, int64_t n) {
  return n <= 16 || (n <= rows / 150 && (n <= 128 || n * rows <= (int64_t)1 << 24));
}

template <typename TX>
static int bf16_dot_launch(const uint16_t* w, int64_t rows, int64_t ldw, const TX* x, int64_t n, float* o,
                           hipStream_t st) {
  const bool vec = n > 0 && n % 4 == 0 && (rows == 1 || ldw % 4 == 0) &&
                   reinterpret_cast<uintptr_t>(w) % (4 * sizeof(uint16_t)) == 0 &&
                   reinterpret_cast<uintptr_t>(x) % (4 * sizeof(TX)) == 0;
  if (bd_short(rows, n))
    hipLaunchKernelGGL(bf16_dot_rows_kernel<TX>, dim3((unsigned)ceil_div(rows, 64)), dim3(64), 0, st, w, rows, ldw, x, n,
                       o);
  else if (rows == 1)
    hipLaunchKernelGGL((vec ? bf16_dot_kernel<1, true, TX> : bf16_dot_kernel<1, false, TX>), dim3(1),
                       dim3(BdShape<1>::kThreads), 0, st, w, rows, ldw, x, n, o);
  else
    hipLaunchKernelGGL((vec ? bf16_dot_kernel<16, true, TX> : bf16_dot_kernel<16, false, TX>),
                       dim3((unsigned)ceil_div(rows, 16)), dim3(BdShape<16>::kThreads), 0, st, w, rows, ldw, x, n, o);
  KH_LAUNCHED();
  return KH_OK;
}

// f32::exp of every element, the same expf_glibc the predictor, SiLU and
// softmax kernels evaluate.
__global__ void expf_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = expf_glibc(x[i]);
}

}  // namespace kh

using namespace kh;

extern "C" int kh_dense_dot_dense(const float* a_dev, int64_t rows, int64_t lda, const float* b_dev,
                                  int64_t n, float* out_dev, void* stream) {
  KH_CHECK_ARG(out_dev && ((a_dev && b_dev) || n == 0 || rows == 0), "null argument");
  KH_CHECK_ARG(rows >= 0 && n >= 0 && lda >= n, "bad shape (rows %lld n %lld lda %lld)",
               (long long)rows, (long long)n, (long long)lda);
  if (rows == 0) return KH_OK;
  const int64_t threads = rows * 16;
  hipLaunchKernelGGL(dense_dot_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     as_stream(stream), a_dev, rows, lda, b_dev, n, out_dev);
  KH_LAUNCHED();
  return KH_OK;
}

extern "C" int kh_sparse_dot_dense(const uint32_t* idx_dev, const float* val_dev, int64_t nnz,
                                   const float* dense_dev, int64_t dense_len, float* out_dev,
                                   void* stream) {
  KH_CHECK_ARG(out_dev && dense_dev && (nnz == 0 || (idx_dev && val_dev)), "null argument");
  KH_CHECK_ARG(nnz >= 0 && dense_len >= 0, "bad shape");
  hipLaunchKernelGGL(sparse_dot_kernel, dim3(1), dim3(256), 0, as_stream(stream), idx_dev, val_dev,
                     nnz, dense_dev, out_dev);
  KH_LAUNCHED();
  return KH_OK;
}

extern "C" int kh_scatter_add(const uint32_t* idx_dev, const float* val_dev, int64_t n,
                              float* dense_dev, int64_t dense_len, float scale, void* stream) {
  KH_CHECK_ARG(dense_dev && (n == 0 || (idx_dev && val_dev)), "null argument");
  KH_CHECK_ARG(n >= 0 && dense_len >= 0, "bad shape");
  if (n == 0) return KH_OK;
  hipLaunchKernelGGL(scatter_add_kernel, dim3(1), dim3(1024), 0, as_stream(stream), idx_dev,
                     val_dev, n, dense_dev, scale);
  KH_LAUNCHED();
  return KH_OK;
}

extern "C" int kh_bf16_from_f32(const float* x_dev, uint16_t* out_dev, int64_t n, void* stream) {
  KH_CHECK_ARG((x_dev && out_dev) || n == 0, "null argument");
  KH_CHECK_ARG(n >= 0, "bad n");
  return ew_launch<EwFromF32>(x_dev, out_dev, n, as_stream(stream));
}

extern "C" int kh_bf16_to_f32(const uint16_t* x_dev, float* out_dev, int64_t n, void* stream) {
  KH_CHECK_ARG((x_dev && out_dev) || n == 0, "null argument");
  KH_CHECK_ARG(n >= 0, "bad n");
  return ew_launch<EwToF32>(x_dev, out_dev, n, as_stream(stream));
}

extern "C" int kh_bf16_update_from_f32(uint16_t* w_dev, const float* delta_dev, int64_t n,
                                       void* stream) {
  KH_CHECK_ARG((w_dev && delta_dev) || n == 0, "null argument");
  KH_CHECK_ARG(n >= 0, "bad n");
  return ew_launch<EwUpdate>(delta_dev, w_dev, n, as_stream(stream));
}

extern "C" int kh_bf16_dot_f32(const uint16_t* w_dev, int64_t rows, int64_t ldw,
                               const float* x_dev, int64_t n, float* out_dev, void* stream) {
  KH_CHECK_ARG(out_dev && ((w_dev && x_dev) || n == 0 || rows == 0), "null argument");
  KH_CHECK_ARG(rows >= 0 && n >= 0 && ldw >= n, "bad shape");
  if (rows == 0) return KH_OK;
  return bf16_dot_launch<float>(w_dev, rows, ldw, x_dev, n, out_dev, as_stream(stream));
}

extern "C" int kh_bf16_full_dot(const uint16_t* a_dev, const uint16_t* b_dev, int64_t n,
                                float* out_dev, void* stream) {
  KH_CHECK_ARG(out_dev && (n == 0 || (a_dev && b_dev)), "null argument");
  KH_CHECK_ARG(n >= 0, "bad n");
  return bf16_dot_launch<uint16_t>(a_dev, 1, n, b_dev, n, out_dev, as_stream(stream));
}

extern "C" int kh_expf(const float* x_dev, float* y_dev, int64_t n, void* stream) {
  KH_CHECK_ARG((x_dev && y_dev) || n == 0, "null argument");
  KH_CHECK_ARG(n >= 0 && n <= ((int64_t)1 << 38), "bad n");
  if (n == 0) return KH_OK;
  hipLaunchKernelGGL(expf_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, as_stream(stream), x_dev, y_dev, n);
  KH_LAUNCHED();
  return KH_OK;
}
