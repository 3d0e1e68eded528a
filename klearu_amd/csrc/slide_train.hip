// slide_train.hip -- SLIDE training on the GPU (gfx950).
//
// Replaces Layer::backward and Layer::rebuild_index
// (crates/klearu-core/src/network/layer.rs:124-233), Network::train_step /
// predict with compute_loss / compute_loss_gradient (network/net.rs:81-230),
// the SGD and Adam updates (optim/sgd.rs, optim/adam.rs), LshIndexTrait::rebuild
// (lsh/index.rs:302-307) and RebuildScheduler (lsh/maintenance.rs:20-98).
//
// The reference trains one example at a time and updates the weights after
// each one, so example e+1's forward pass reads the weights example e wrote:
// the examples of a batch are a chain.  Each example is a short sequence of
// kernels on one stream; the parallel work is inside an example (the
// neurons of a layer, the dimensions of a gradient, the weights of an update).
// Prediction writes no weights, so its examples are rows of one batch: the
// forward kernels take a row per block (net_predict_rows).
//
// Every f32 operation is the reference's, in its order: sums over the active
// list run sequentially in the list's order (the Jacobian and grad_input
// sums keep one lane per output, each lane a chain), the softmax denominator
// is the reference's sequential sum computed by exact_seq_sum, and no
// multiply-add is contracted (the library builds with -ffp-contract=off).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "chain_add.hpp"
#include "exact_sum.hpp"
#include "gather.hpp"
#include "entry_sum.hpp"
#include "slide_internal.hpp"

namespace kh {

constexpr int kTrThreads = 256;
constexpr int kTrMaxLabels = 1024;   // labels of one example
constexpr int kTrLdsNz = 8192;       // staged input nonzeros at most (beyond: read from global)
constexpr int kTrMaxNnz = 4096;      // stored entries of one sparse example
constexpr int kSmCH = 64, kSmM = 128;  // exact softmax sum: 8192 terms per pass

struct OptArgs {
  int kind;       // KH_OPT_SGD / KH_OPT_ADAM
  float lr, momentum, b1, b2, eps, c1, c2;
  float* st_w1;   // SGD momentum / Adam first moments [n][dim]
  float* st_w2;   // Adam second moments [n][dim]
  float* st_b1;   // [n]
  float* st_b2;   // [n]
};

// f32::powi with a run-time exponent: the __powisf2 builtin of Rust's
// compiler-builtins (src/float/pow.rs), square-and-multiply from the low bit.
static float powi_f32(float a, int32_t b) {
  const bool recip = b < 0;
  uint32_t p = recip ? 0u - static_cast<uint32_t>(b) : static_cast<uint32_t>(b);
  float mul = 1.0f;
  for (;;) {
    if (p & 1u) mul = mul * a;
    p >>= 1;
    if (p == 0) break;
    a = a * a;
  }
  return recip ? 1.0f / mul : mul;
}

static OptArgs opt_args(const kh_slide_layer* l, double lr, uint64_t step) {
  OptArgs o{};
  o.kind = l->opt;
  o.lr = static_cast<float>(lr);
  o.momentum = l->momentum;
  o.b1 = l->beta1;
  o.b2 = l->beta2;
  o.eps = l->eps;
  // Adam::update (adam.rs:38-47): step.max(1), `step as i32`
  const uint64_t s = step < 1 ? 1 : step;
  const int32_t si = static_cast<int32_t>(static_cast<uint32_t>(s));
  o.c1 = 1.0f - powi_f32(l->beta1, si);
  o.c2 = 1.0f - powi_f32(l->beta2, si);
  o.st_w1 = l->st_w1;
  o.st_w2 = l->st_w2;
  o.st_b1 = l->st_b1;
  o.st_b2 = l->st_b2;
  return o;
}

// activation_derivative (layer.rs:266-283)
__device__ __forceinline__ float act_deriv(float pre, float post, int act) {
  if (act == KH_ACT_RELU) return pre > 0.0f ? 1.0f : 0.0f;
  if (act == KH_ACT_SIGMOID) return post * (1.0f - post);
  if (act == KH_ACT_TANH) return 1.0f - post * post;
  return 1.0f;
}

// apply_activation (layer.rs:250-261)
__device__ __forceinline__ float act_apply(float z, int act) {
  if (act == KH_ACT_RELU) return fmaxf(z, 0.0f);
  if (act == KH_ACT_SIGMOID) return sigmoid_ref(z);
  if (act == KH_ACT_TANH) return tanhf(z);
  return z;
}

// One optimizer step of a parameter (Sgd::update, sgd.rs:28-56; Adam::update,
// adam.rs:50-76); s1/s2 its state slots.
__device__ __forceinline__ float opt_step(float w, float g, float* s1, float* s2, const OptArgs& o) {
  if (o.kind == KH_OPT_ADAM) {
    const float m = o.b1 * *s1 + (1.0f - o.b1) * g;
    const float gg = (1.0f - o.b2) * g;
    const float v = o.b2 * *s2 + gg * g;
    *s1 = m;
    *s2 = v;
    const float mh = m / o.c1;
    const float vh = v / o.c2;
    return w - (o.lr * mh) / (sqrtf(vh) + o.eps);
  }
  if (o.momentum > 0.0f) {
    const float v = o.momentum * *s1 - o.lr * g;
    *s1 = v;
    return w + v;
  }
  return w - o.lr * g;
}

// Nonzeros of each dense row in ascending order: block r's list starts at
// nzi/nzv + r * stride and runs over xoff[2r] .. xoff[2r + 1].
// Dropping zero terms leaves every sequential sum over the vector unchanged
// (x + 0 == x; a zero partial sum only changes the sign of zero), so hashes
// and neuron sums over the list equal the reference's dense loops.
__global__ __launch_bounds__(1024) void tr_stage_nz_kernel(const float* __restrict__ x, int dim,
                                                           int64_t ldx, int64_t stride,
                                                           uint32_t* __restrict__ nzi,
                                                           float* __restrict__ nzv,
                                                           int64_t* __restrict__ xoff) {
  __shared__ int wsum[16];
  __shared__ int s_total;
  const int64_t row = blockIdx.x;
  x += row * ldx;
  nzi += row * stride;
  nzv += row * stride;
  int base = 0;
  for (int c0 = 0; c0 < dim; c0 += blockDim.x) {
    const int d = c0 + threadIdx.x;
    const float v = d < dim ? x[d] : 0.0f;
    const int nz = v != 0.0f ? 1 : 0;
    const int pos = block_excl_scan(nz, wsum, &s_total) + base;
    if (nz) {
      nzi[pos] = static_cast<uint32_t>(d);
      nzv[pos] = v;
    }
    base += s_total;
  }
  if (threadIdx.x == 0) {
    xoff[2 * row] = row * stride;
    xoff[2 * row + 1] = row * stride + base;
  }
}

// Example::features.to_dense() (tensor/sparse.rs:77-83) of CSR rows row0 +
// blockIdx.x: later stored entries overwrite earlier ones at the same index, so
// after a sort by (index, position) the last entry of each index is the value;
// the nonzero values in ascending index order become the row's staged list
// (laid out as tr_stage_nz_kernel's), and x_dense, when given (one row), gets
// them (the previous row's entries are cleared first).  Entries with index >=
// dim are skipped (to_dense would panic on them).  A block per row, bound by
// latency: a row whose entries are already in index order (as LIBSVM files and
// to_sparse give them) is not sorted, and its values come with its indices: one row
// of 75 entries takes 3.7 us; 7.8 when every row was sorted first.
__global__ __launch_bounds__(1024) void tr_stage_csr_kernel(
    const int64_t* __restrict__ xoff, const uint32_t* __restrict__ xidx,
    const float* __restrict__ xval, int64_t row0, int dim, int64_t stride,
    uint32_t* __restrict__ nzi, float* __restrict__ nzv, int64_t* __restrict__ nzoff,
    float* __restrict__ x_dense) {
  __shared__ uint64_t key[kTrMaxNnz];
  __shared__ float val[kTrMaxNnz];
  __shared__ int wsum[16];
  __shared__ int s_total;
  const int64_t out = static_cast<int64_t>(blockIdx.x) * stride;
  const int64_t row = row0 + blockIdx.x;
  nzi += out;
  nzv += out;
  const int64_t a = xoff[row], b = xoff[row + 1];
  const int old = x_dense ? static_cast<int>(nzoff[1]) : 0;
  const int cnt = static_cast<int>(min<int64_t>(b - a, kTrMaxNnz));
  int P = 1;
  while (P < cnt) P <<= 1;
  for (int i = threadIdx.x; i < P; i += blockDim.x) {
    key[i] = i < cnt ? (static_cast<uint64_t>(xidx[a + i]) << 32) | static_cast<uint32_t>(i) : ~0ull;
    val[i] = i < cnt ? xval[a + i] : 0.0f;
  }
  for (int i = threadIdx.x; i < old; i += blockDim.x) x_dense[nzi[i]] = 0.0f;
  __syncthreads();
  int unsorted = 0;
  for (int i = threadIdx.x; i + 1 < cnt; i += blockDim.x) unsorted |= key[i] > key[i + 1] ? 1 : 0;
  for (int k = __syncthreads_or(unsorted) ? 2 : P + 1; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < P; i += blockDim.x) {
        const int ixj = i ^ j;
        if (ixj > i) {
          const uint64_t x = key[i], y = key[ixj];
          if ((x > y) == ((i & k) == 0)) {
            key[i] = y;
            key[ixj] = x;
          }
        }
      }
      __syncthreads();
    }
  }
  int base = 0;
  for (int c0 = 0; c0 < P; c0 += blockDim.x) {
    const int i = c0 + threadIdx.x;
    int keep = 0;
    uint32_t idx = 0;
    float v = 0.0f;
    if (i < cnt) {
      idx = static_cast<uint32_t>(key[i] >> 32);
      const bool last = i + 1 == cnt || static_cast<uint32_t>(key[i + 1] >> 32) != idx;
      v = val[static_cast<uint32_t>(key[i])];
      keep = last && v != 0.0f && idx < static_cast<uint32_t>(dim);
    }
    const int pos = block_excl_scan(keep, wsum, &s_total) + base;
    if (keep) {
      nzi[pos] = idx;
      nzv[pos] = v;
      if (x_dense) x_dense[idx] = v;
    }
    base += s_total;
  }
  if (threadIdx.x == 0) {
    nzoff[2 * blockIdx.x] = out;
    nzoff[2 * blockIdx.x + 1] = out + base;
  }
}

// Neuron::forward for one example's active list over row-major weights: a wave per
// neuron, lanes over the entries, so that up to kTwEntries scattered weights are in
// flight at once (a thread per neuron had five rounds of sixteen for 75 entries, in
// two blocks: 14.6 us for 128 neurons of 8192 inputs; 4.3 us here).  The products pass
// through the wave's own LDS to be added in order by every lane alike.
constexpr int kTwEntries = 256;
__global__ __launch_bounds__(kTrThreads) void tr_neuron_wave_kernel(
    const float* __restrict__ W, const float* __restrict__ bias, int dim, const uint32_t* __restrict__ nzi,
    const float* __restrict__ nzv, const int64_t* __restrict__ xoff, const uint32_t* __restrict__ aids,
    const int32_t* __restrict__ alen, int cap, int act, float* __restrict__ pre, float* __restrict__ post,
    float* __restrict__ dense) {
  constexpr int U = kTwEntries / 64, kWaves = kTrThreads / 64, Q = 4;   // Q: float4 read ahead
  __shared__ __align__(16) float prod[kWaves][kTwEntries];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = min(alen[0], cap);
  const int64_t first = xoff[0];
  const int nnz = static_cast<int>(xoff[1] - first);
  nzi += first;
  nzv += first;
  for (int a = blockIdx.x * kWaves + wave; a < n; a += gridDim.x * kWaves) {
    const uint32_t id = aids[a];
    const float b = bias[id];
    const float* __restrict__ w = W + static_cast<size_t>(id) * dim;
    float s = -0.0f;
    for (int e0 = 0; e0 < nnz; e0 += kTwEntries) {
      const int m = min(kTwEntries, nnz - e0);
      uint32_t d[U];
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + min(64 * u + lane, m - 1);
        d[u] = nzi[e];
        v[u] = nzv[e];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = __fmul_rn(w[d[u]], v[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) prod[wave][64 * u + lane] = 64 * u + lane < m ? v[u] : -0.0f;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's products are in LDS
      const float4* p4 = reinterpret_cast<const float4*>(prod[wave]);
      const int groups = (m + 4 * Q - 1) / (4 * Q);
      float4 r[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) r[q] = p4[q];
      for (int g = 0; g < groups; ++g) {
        float4 nx[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) nx[q] = p4[min(g + 1, groups - 1) * Q + q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          s = __fadd_rn(s, r[q].x);
          s = __fadd_rn(s, r[q].y);
          s = __fadd_rn(s, r[q].z);
          s = __fadd_rn(s, r[q].w);
        }
        asm volatile("" : "+v"(s));
#pragma unroll
        for (int q = 0; q < Q; ++q) r[q] = nx[q];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the next products
    }
    if (lane == 0) {
      const float z = __fadd_rn(s, b);
      pre[a] = z;
      if (act != KH_ACT_SOFTMAX) {
        const float r = act_apply(z, act);
        post[a] = r;
        dense[id] = r;
      }
    }
  }
}

// Neuron::forward (neuron.rs:47-62) for each sample's active list (row
// blockIdx.y: aids, pre and post rows of `cap` entries, dense rows of
// dense_ld): the sequential sum of w*x over the staged nonzeros, + bias; then
// the activation (not softmax) into post and the dense activation vector.
// TRANS: W is the transposed copy [dim][n] (n = dim_or_n), whose row of one
// input holds the weights of every active neuron; otherwise [n][dim].  Lists of
// up to lds_nz entries (the dynamic LDS holds that many) are read from LDS.
// 128 rows of 157 nonzeros, 256 of 1024 neurons each: 17.4 us, 22.4 with each sixteen
// loads waited for before the next.
template <bool TRANS>
__global__ __launch_bounds__(kTrThreads) void tr_neuron_kernel(
    const float* __restrict__ W, const float* __restrict__ bias, int dim, int dim_or_n, int lds_nz,
    const uint32_t* __restrict__ nzi, const float* __restrict__ nzv,
    const int64_t* __restrict__ xoff, const uint32_t* __restrict__ aids,
    const int32_t* __restrict__ alen, int cap, int act, float* __restrict__ pre,
    float* __restrict__ post, float* __restrict__ dense, int64_t dense_ld) {
  extern __shared__ unsigned char smem[];
  const int64_t row = blockIdx.y;
  const int n = min(alen[row], cap);
  if (static_cast<int>(blockIdx.x * blockDim.x) >= n) return;
  aids += row * cap;
  pre += row * cap;
  post += row * cap;
  dense += row * dense_ld;
  const int64_t first = xoff[2 * row];
  const int nnz = static_cast<int>(xoff[2 * row + 1] - first);
  nzi += first;
  nzv += first;
  const bool in_lds = nnz <= lds_nz;
  const bool fit = TRANS && offsets_fit(dim, dim_or_n);
  uint32_t* si = reinterpret_cast<uint32_t*>(smem);
  float* sv = reinterpret_cast<float*>(smem + sizeof(uint32_t) * lds_nz);
  if (in_lds) {
    const int npad = entries_padded(nnz);
    for (int i = threadIdx.x; i < npad; i += blockDim.x) {
      si[i] = i < nnz ? nzi[i] * (fit ? (uint32_t)dim_or_n : 1u) : 0u;
      sv[i] = i < nnz ? nzv[i] : 0.0f;
    }
    __syncthreads();
  }
  for (int a = blockIdx.x * blockDim.x + threadIdx.x; a < n; a += gridDim.x * blockDim.x) {
    const uint32_t id = aids[a];
    const float* w = TRANS ? W + id : W + static_cast<size_t>(id) * dim_or_n;
    const size_t step = TRANS ? dim_or_n : 1;
    float s = -0.0f;
    if (in_lds && nnz && fit) {
      s = sum_entries(si, sv, nnz, [&](uint32_t q) { return weight_at(W, id + q); });
    } else if (in_lds && nnz) {
      s = sum_entries(si, sv, nnz, [&](uint32_t d) { return w[d * step]; });
    } else {
      for (int e = 0; e < nnz; ++e) s = s + w[nzi[e] * step] * nzv[e];
    }
    const float z = s + bias[id];
    pre[a] = z;
    if (act != KH_ACT_SOFTMAX) {
      const float r = act_apply(z, act);
      post[a] = r;
      dense[id] = r;
    }
  }
}

// apply_softmax (layer.rs:286-308) over each row's active list (block r: rows
// of `cap` entries, dense rows of dense_ld) in its order: max, exp(z - max) with
// glibc's expf, the sequential sum, then e / sum (or 1/n when the sum is not
// positive).  Lists of up to kPass entries stay in registers (all loads in
// flight); longer ones go through `post` in passes.  The sum: a plain chain of
// adds up to kSmChain entries (2.5 us at 512), exact_seq_sum beyond.  Sixteen
// waves, because the exps are double-precision chains: 4400 entries 16.0 -> 10.2 us
// against four waves, 32 entries in 128 rows 21.6 -> 9.9 us.
constexpr int kSmThreads = 1024;
constexpr int kSmChain = 512;
__global__ __launch_bounds__(kSmThreads) void tr_softmax_kernel(const float* __restrict__ pre,
                                                                const uint32_t* __restrict__ aids,
                                                                const int32_t* __restrict__ alen,
                                                                int cap, float* __restrict__ post,
                                                                float* __restrict__ dense,
                                                                int64_t dense_ld) {
  constexpr int kPass = kSmCH * kSmM;
  constexpr int kPer = kPass / kSmThreads;
  constexpr int kWaves = kSmThreads / 64;
  __shared__ EsLds<kSmCH, kSmM> es;
  __shared__ float red[kWaves];
  __shared__ uint64_t s_tab[32];  // kExp2Tab: the exps' table lookups stay in LDS
  const int64_t row = blockIdx.x;
  const int n = min(alen[row], cap);
  if (n <= 0) return;
  pre += row * cap;
  aids += row * cap;
  post += row * cap;
  if (dense) dense += row * dense_ld;
  if (threadIdx.x < 32) s_tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  float v[kPer];
  float mx = -INFINITY;
  if (n <= kPass) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) v[k] = pre[min(k * kSmThreads + static_cast<int>(threadIdx.x), n - 1)];
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      v[k] = k * kSmThreads + static_cast<int>(threadIdx.x) < n ? v[k] : -INFINITY;
#pragma unroll
    for (int k = 0; k < kPer; ++k) mx = fmaxf(mx, v[k]);
  } else {
    for (int a = threadIdx.x; a < n; a += blockDim.x) mx = fmaxf(mx, pre[a]);
  }
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = red[0];
  for (int i = 1; i < kWaves; ++i) mx = fmaxf(mx, red[i]);
  float s = -0.0f;
  if (n <= kPass) {
    const bool chain = n <= kSmChain;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int a = k * kSmThreads + threadIdx.x;
      v[k] = a < n ? expf_glibc_t(v[k] - mx, s_tab) : -0.0f;
      if (!chain) es.TP[es_slot<kSmCH, kSmM>(a)] = v[k];
    }
    if (chain) {
      static_assert(kSmChain <= kSmThreads, "one term per thread");
      if (threadIdx.x < kSmChain) es.TP[threadIdx.x] = v[0];   // -0.0 past n
      __syncthreads();
      const float4* q = reinterpret_cast<const float4*>(es.TP);
#pragma unroll 1
      for (int g = 0; g < n; g += 32) s = chain_add_static<8, 1>(q + g / 4, s);   // every wave: the same sum
    } else {
      __syncthreads();
      s = exact_seq_sum<kWaves, kSmCH, kSmM>(n, s, es);
    }
    const float u = 1.0f / static_cast<float>(n);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int a = k * kSmThreads + threadIdx.x;
      if (a < n) {
        const float r = s > 0.0f ? v[k] / s : u;
        post[a] = r;
        if (dense) dense[aids[a]] = r;
      }
    }
    return;
  }
  for (int a = threadIdx.x; a < n; a += blockDim.x) post[a] = expf_glibc_t(pre[a] - mx, s_tab);
  __syncthreads();
  for (int c0 = 0; c0 < n; c0 += kPass) {
    const int cnt = min(kPass, n - c0);
    for (int i = threadIdx.x; i < kPass; i += blockDim.x)
      es.TP[es_slot<kSmCH, kSmM>(i)] = i < cnt ? post[c0 + i] : -0.0f;
    __syncthreads();
    s = exact_seq_sum<kWaves, kSmCH, kSmM>(cnt, s, es);
  }
  const float u = 1.0f / static_cast<float>(n);
  for (int a = threadIdx.x; a < n; a += blockDim.x) {
    const float r = s > 0.0f ? post[a] / s : u;
    post[a] = r;
    if (dense) dense[aids[a]] = r;
  }
}

// compute_loss and compute_loss_gradient (net.rs:180-230) of one example at
// the last layer's active entries: go[a] = activations[id] minus 1/|labels|
// per occurrence of id among the labels (all zero without labels); lg[a] =
// go * activation_derivative unless the layer is softmax (the Jacobian kernel
// follows).  One thread adds the example's loss to *loss_total, so the total
// is the reference's sequential f32 sum over the batch.  One block (the losses
// found are its own): sixteen waves, as each pass over the list is two round trips.
// 4470 outputs: 4.0 us, 6.4 with four waves.
constexpr int kLossThreads = 1024;
__global__ __launch_bounds__(kLossThreads) void tr_loss_grad_kernel(
    const float* __restrict__ pre, const float* __restrict__ post,
    const uint32_t* __restrict__ aids, const int32_t* __restrict__ alen, int cap, int act,
    const float* __restrict__ dense, const uint32_t* __restrict__ labels, int nl,
    float* __restrict__ go, float* __restrict__ lg, float* __restrict__ loss_total) {
  __shared__ int found[kTrMaxLabels];
  __shared__ uint32_t lab[kTrMaxLabels];
  const int n = min(alen[0], cap);
  for (int l = threadIdx.x; l < nl; l += blockDim.x) {
    found[l] = 0;
    lab[l] = labels[l];
  }
  __syncthreads();
  const float w = nl > 0 ? 1.0f / static_cast<float>(nl) : 0.0f;
  for (int a = threadIdx.x; a < n; a += blockDim.x) {
    const uint32_t id = aids[a];
    float g = nl > 0 ? post[a] : 0.0f;
    for (int l = 0; l < nl; ++l)
      if (lab[l] == id) {
        g = g - w;
        found[l] = 1;
      }
    go[a] = g;
    if (act != KH_ACT_SOFTMAX) lg[a] = g * act_deriv(pre[a], post[a], act);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float loss = 0.0f;
    if (nl > 0) {
      const float eps = 1e-7f;
      for (int l = 0; l < nl; ++l) {
        const float prob = found[l] ? fmaxf(dense[lab[l]], eps) : eps;
        loss = loss - logf(prob);
      }
      loss = loss / static_cast<float>(nl);
    }
    *loss_total = *loss_total + loss;
  }
}

// The softmax branch of Layer::backward (layer.rs:141-175): output i's local
// gradient is the sequential sum over j (from +0.0) of go_j*s_j*(1-s_j) when
// j == i, else go_j*(-s_i*s_j).  The chain of n dependent adds bounds it.  A block
// owns 32 outputs, one chain per lane of wave 0; the terms, two rounded products
// each, are formed in LDS by six waves, which read (s, go) straight into registers
// kJAhead chunks early.  Wave 4 only keeps the barriers: a block's waves go to the
// SIMDs in turn, so wave 0 shares its SIMD with no producer.  Half a wave of
// chains per block halves the LDS traffic per CU (64 chains would move 96 KB a
// chunk, as long as the adds take) and spreads a list over more CUs.  Steps past
// the list are -0.0, so the last chunk needs no loop of its own.
// 4470 outputs: 16.4 us; 32.5 with 64 chains, three producer waves and a loader
// wave.
constexpr int kJc = 32;                      // chains per block
constexpr int kJStep = 192;                  // steps per chunk
constexpr int kJProd = 6;                    // producer waves (1-3 and 5-7)
constexpr int kJThreads = 512;
constexpr int kJAhead = 2;
constexpr int kJPer = kJStep / 4 / (2 * kJProd);   // quads per producer half wave and chunk
constexpr int kJBlocks = 256;                // grid (groups of 32 outputs are strided over it)
static_assert(kJPer * 2 * kJProd * 4 == kJStep, "whole quads per producer");
constexpr int kJPad = 4;                     // floats past a list that the quad loads may touch

__device__ __forceinline__ float jac_off(float gj, float sj, float nsi) { return gj * (nsi * sj); }

__global__ __launch_bounds__(kJThreads) void tr_softmax_jacobian_kernel(
    const float* __restrict__ s, const float* __restrict__ go, const int32_t* __restrict__ alen,
    int cap, float* __restrict__ lg) {
  using Lds = ChainLds<kJStep, kJc>;
  __shared__ Lds lds;
  const int n = min(alen[0], cap);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nch = (n + kJStep - 1) / kJStep;
  const bool prod = wave != 0 && wave != 4;
  const int p = 2 * (wave < 4 ? wave - 1 : wave - 2) + (lane >> 5);  // producer half wave
  for (int i0 = blockIdx.x * kJc; i0 < n; i0 += gridDim.x * kJc) {
    const int i = min(i0 + (lane & (kJc - 1)), n - 1);
    const float si = s[i], gi = go[i];
    const float nsi = -si;
    const float dterm = (gi * si) * (1.0f - si);  // the diagonal term, j == i
    float4 sv[kJAhead][kJPer], gv[kJAhead][kJPer];
    // quads p, p + 2 kJProd, ... of chunk c (past the list: its last quad)
    auto fetch = [&](int c, int u) {
#pragma unroll
      for (int e = 0; e < kJPer; ++e) {
        const int q = min(c * (kJStep / 4) + p + 2 * kJProd * e, (n - 1) / 4);
        sv[u][e] = reinterpret_cast<const float4*>(s)[q];
        gv[u][e] = reinterpret_cast<const float4*>(go)[q];
      }
    };
    lds_barrier();  // the group before is consumed
    if (prod) {
#pragma unroll
      for (int u = 0; u < kJAhead; ++u) fetch(u, u);
    }
    const float r = chain_run<kJAhead>(lds, nch, 0.0f, [&](int c, int u) {
#pragma unroll
      for (int e = 0; e < kJPer; ++e) {
        const int q = p + 2 * kJProd * e;
        const int j = c * kJStep + 4 * q;
        const int d = i0 + (lane & (kJc - 1)) - j;   // step of the diagonal
        const float4 a = sv[u][e], g = gv[u][e];
        float4 t = make_float4(jac_off(g.x, a.x, nsi), jac_off(g.y, a.y, nsi), jac_off(g.z, a.z, nsi),
                               jac_off(g.w, a.w, nsi));
        t.x = d == 0 ? dterm : j < n ? t.x : -0.0f;
        t.y = d == 1 ? dterm : j + 1 < n ? t.y : -0.0f;
        t.z = d == 2 ? dterm : j + 2 < n ? t.z : -0.0f;
        t.w = d == 3 ? dterm : j + 3 < n ? t.w : -0.0f;
        lds.q[c & 1][q * Lds::kStride + (lane & (kJc - 1))] = t;
      }
      fetch(c + kJAhead, u);
    }, wave == 4);
    if (wave == 0 && lane < kJc && i0 + lane < n) lg[i0 + lane] = r;
  }
}

// Local gradients of a layer from the gradient w.r.t. its output: go = the
// entry at the neuron's id (0 past the length); non-softmax layers get
// lg = go * activation_derivative(pre, activations[id]); softmax layers keep
// go for the Jacobian.
__global__ __launch_bounds__(kTrThreads) void tr_local_grad_kernel(
    const uint32_t* __restrict__ aids, const int32_t* __restrict__ alen, int cap,
    const float* __restrict__ pre, const float* __restrict__ dense, int act,
    const float* __restrict__ grad_out, int64_t grad_len, float* __restrict__ go,
    float* __restrict__ lg) {
  const int n = min(alen[0], cap);
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= n) return;
  const uint32_t id = aids[a];
  const float g = static_cast<int64_t>(id) < grad_len ? grad_out[id] : 0.0f;
  if (act == KH_ACT_SOFTMAX)
    go[a] = g;
  else
    lg[a] = g * act_deriv(pre[a], dense[id], act);
}

// grad_input[j] = sum over the active list (in order, from +0.0) of
// lg[a] * w[id_a][j], with the weights before this example's update
// (layer.rs:203-207).  Each j is one chain of |A| dependent adds; a block owns
// kGc columns, one chain per lane of wave 0, and the other waves gather the
// products of kGStep active rows a chunk into LDS, kGAhead chunks of row pieces
// (and the ids of as many more) in flight: 16 blocks at 128 columns have to pull
// the rows at the chains' pace.  4470 rows of 128: 17.0 us, 25.5 with
// 1024-row chunks and one chunk in flight.
// VEC: dim a multiple of 4.
constexpr int kGc = 8;          // columns (chains) per block
constexpr int kGStep = 128;     // active rows per chunk
constexpr int kGAhead = 8;
constexpr int kGThreads = 64 + kGStep * (kGc / 4);

template <bool VEC>
__global__ __launch_bounds__(kGThreads) void tr_grad_input_kernel(
    const float* __restrict__ W, int dim, const uint32_t* __restrict__ aids,
    const int32_t* __restrict__ alen, int cap, const float* __restrict__ lg,
    float* __restrict__ gi) {
  using Lds = ChainLds<kGStep, kGc>;
  __shared__ Lds lds;
  const int n = min(alen[0], cap);
  const int j0 = blockIdx.x * kGc;
  const int nch = (n + kGStep - 1) / kGStep;
  const bool prod = threadIdx.x >= 64;
  const int pt = static_cast<int>(threadIdx.x) - 64;
  const int q = pt & (kGc / 4 - 1), e = pt / (kGc / 4);   // column quad, row within the chunk
  const int jq = j0 + 4 * q;
  uint32_t id[kGAhead];                                   // row of the chunk kGAhead past the slot's
  float4 w[kGAhead];
  float l[kGAhead];
  auto ids = [&](int c, int u) { id[u] = aids[min(c * kGStep + e, n - 1)]; };
  auto fetch = [&](int c, int u) {
    const float* __restrict__ r = W + static_cast<size_t>(id[u]) * dim;
    if constexpr (VEC)
      w[u] = *reinterpret_cast<const float4*>(r + min(jq, dim - 4));
    else
      w[u] = make_float4(r[min(jq, dim - 1)], r[min(jq + 1, dim - 1)], r[min(jq + 2, dim - 1)], r[min(jq + 3, dim - 1)]);
    l[u] = lg[min(c * kGStep + e, n - 1)];
  };
  if (prod && nch > 0) {
#pragma unroll
    for (int u = 0; u < kGAhead; ++u) ids(u, u);
#pragma unroll
    for (int u = 0; u < kGAhead; ++u) fetch(u, u);
#pragma unroll
    for (int u = 0; u < kGAhead; ++u) ids(u + kGAhead, u);
  }
  const float r = chain_run<kGAhead>(lds, nch, 0.0f, [&](int c, int u) {
    const bool on = c * kGStep + e < n;
    float* d = reinterpret_cast<float*>(&lds.q[c & 1][(e >> 2) * Lds::kStride + 4 * q]) + (e & 3);
    d[0] = on ? l[u] * w[u].x : -0.0f;
    d[4] = on ? l[u] * w[u].y : -0.0f;
    d[8] = on ? l[u] * w[u].z : -0.0f;
    d[12] = on ? l[u] * w[u].w : -0.0f;
    fetch(c + kGAhead, u);
    ids(c + 2 * kGAhead, u);
  });
  if (threadIdx.x < kGc && j0 + static_cast<int>(threadIdx.x) < dim) gi[j0 + threadIdx.x] = r;
}

// Optimizer::update of every active neuron (layer.rs:209-222): grad_weights[j]
// = lg * x[j] over all dim inputs (zeros included: momentum and Adam state
// move every step), grad_bias = lg.  The transposed copy follows the rows.
// Bound by latency up to some ten MB of weights and state, so the active rows are
// one run of na * dim weights cut into tiles of kUTile (a block of a row of its own
// would leave half its threads idle at dim 128), and a thread has its kUPer weights,
// states and inputs in flight together.  STATES: state arrays of the optimizer (Adam 2,
// momentum 1, plain SGD 0).  The last blocks, which get the fewest tiles, take the biases.
// 128 rows of 8192 and 4470 rows of 128 (Adam): 14.2 us together, 16.5 with a block per row.
constexpr int kUPer = 4;
constexpr int kUTile = kTrThreads * kUPer;
// Sixteen blocks per CU, twice what runs at once: 128 rows of 135909 67 us, 76 with 2048 (70 with a
// block per row and 2048 columns); tiles beyond are strided over them.
constexpr int kUBlocks = 4096;
template <int STATES>
__global__ __launch_bounds__(kTrThreads) void tr_update_kernel(
    float* __restrict__ W, float* __restrict__ WTN, float* __restrict__ bias, int n, int dim,
    const uint32_t* __restrict__ aids, const int32_t* __restrict__ alen, int cap,
    const float* __restrict__ lg, const float* __restrict__ x, OptArgs o) {
  const int na = min(alen[0], cap);
  const int64_t total = static_cast<int64_t>(na) * dim;
  const uint32_t udim = static_cast<uint32_t>(dim);
  for (int64_t e0 = static_cast<int64_t>(blockIdx.x) * kUTile; e0 < total; e0 += static_cast<int64_t>(gridDim.x) * kUTile) {
    const int64_t a0 = e0 / dim;
    const uint32_t j0 = static_cast<uint32_t>(e0 - a0 * dim);
    float w[kUPer], s1[kUPer], s2[kUPer], xv[kUPer], g[kUPer];
    uint32_t id[kUPer], jj[kUPer];
    size_t at[kUPer];
    bool on[kUPer];
#pragma unroll
    for (int u = 0; u < kUPer; ++u) {  // clamped, unconditional: every load is in flight
      const uint32_t off = j0 + threadIdx.x + u * kTrThreads;
      const uint32_t r = off / udim;
      on[u] = a0 + r < na;
      const int64_t a = min(a0 + static_cast<int64_t>(r), static_cast<int64_t>(na) - 1);
      jj[u] = off - r * udim;
      id[u] = aids[a];
      g[u] = lg[a];
      xv[u] = x[jj[u]];
    }
#pragma unroll
    for (int u = 0; u < kUPer; ++u) {
      on[u] = on[u] && id[u] < static_cast<uint32_t>(n);
      at[u] = static_cast<size_t>(min(id[u], static_cast<uint32_t>(n) - 1)) * dim + jj[u];
      w[u] = W[at[u]];
      s1[u] = STATES > 0 ? o.st_w1[at[u]] : 0.0f;
      s2[u] = STATES > 1 ? o.st_w2[at[u]] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kUPer; ++u) {
      const float nw = opt_step(w[u], g[u] * xv[u], &s1[u], &s2[u], o);
      if (on[u]) {
        W[at[u]] = nw;
        if (STATES > 0) o.st_w1[at[u]] = s1[u];
        if (STATES > 1) o.st_w2[at[u]] = s2[u];
        if (WTN) WTN[static_cast<size_t>(jj[u]) * n + id[u]] = nw;
      }
    }
  }
  for (int a = (gridDim.x - 1 - blockIdx.x) * kTrThreads + threadIdx.x; a < na; a += gridDim.x * kTrThreads) {
    const uint32_t id = aids[a];
    if (id >= static_cast<uint32_t>(n)) continue;
    bias[id] = opt_step(bias[id], lg[a], STATES > 0 ? o.st_b1 + id : nullptr, STATES > 1 ? o.st_b2 + id : nullptr, o);
  }
}

// Local gradients -> (grad_input) -> update of one layer for one example.
// x: the layer's dense input; post: activations in list order (softmax only).
// keep_wtn: write updated rows into the transposed copy too (scattered
// 4-byte stores, one per weight); a network step instead re-transposes once
// after the whole batch (wtn_refresh).
static int layer_backward_launch(kh_slide_layer* l, const float* x, const uint32_t* aids,
                                 const int32_t* alen, int cap, const float* pre,
                                 const float* post, const float* dense, const float* grad_out,
                                 int64_t grad_len, bool lg_ready, float* go, float* lg,
                                 const OptArgs& o, float* gi, bool keep_wtn, hipStream_t st) {
  const unsigned ab = static_cast<unsigned>(ceil_div(cap, kTrThreads));
  if (!lg_ready) {
    hipLaunchKernelGGL(tr_local_grad_kernel, dim3(ab), dim3(kTrThreads), 0, st, aids, alen, cap,
                       pre, dense, l->act, grad_out, grad_len, go, lg);
    KH_LAUNCHED();
  }
  if (l->act == KH_ACT_SOFTMAX) {
    hipLaunchKernelGGL(tr_softmax_jacobian_kernel, dim3((unsigned)std::min(ceil_div(cap, kJc), kJBlocks)),
                       dim3(kJThreads), 0, st, post, go, alen, cap, lg);
    KH_LAUNCHED();
  }
  if (gi) {
    hipLaunchKernelGGL((l->dim % 4 == 0 ? tr_grad_input_kernel<true> : tr_grad_input_kernel<false>),
                       dim3((unsigned)ceil_div(l->dim, kGc)), dim3(kGThreads), 0, st, l->w, l->dim, aids, alen, cap, lg, gi);
    KH_LAUNCHED();
  }
  const int64_t tiles = ceil_div(static_cast<int64_t>(cap) * l->dim, static_cast<int64_t>(kUTile));
  auto update = o.kind == KH_OPT_ADAM ? tr_update_kernel<2> : o.momentum > 0.0f ? tr_update_kernel<1> : tr_update_kernel<0>;
  hipLaunchKernelGGL(update, dim3((unsigned)std::clamp<int64_t>(tiles, 1, kUBlocks)), dim3(kTrThreads), 0, st, l->w,
                     keep_wtn ? l->wtn : nullptr, l->bias, l->n, l->dim, aids, alen, cap, lg, x, o);
  KH_LAUNCHED();
  return KH_OK;
}

// The transposed copy of a non-softmax layer rebuilt from the weights.
static int wtn_refresh(kh_slide_layer* l, hipStream_t st) {
  if (!l->wtn) return KH_OK;
  hipLaunchKernelGGL(transpose_kernel<float>, dim3(ceil_div(l->dim, 32), ceil_div(l->n, 32)), dim3(256),
                     0, st, l->w, l->n, l->dim, l->wtn);
  KH_LAUNCHED();
  return KH_OK;
}

}  // namespace kh

using namespace kh;

// ======================================================================== scheduler
static uint64_t sched_interval(const kh_rebuild_scheduler* s) {
  // (base as f64 * (decay * count as f64).exp()) as usize, then .max(1)
  const double v = static_cast<double>(s->base_interval) *
                   std::exp(s->decay * static_cast<double>(s->rebuild_count));
  uint64_t n;
  if (!(v > 0.0)) n = 0;                              // NaN and <= 0 saturate to 0
  else if (v >= 18446744073709551616.0) n = UINT64_MAX;
  else n = static_cast<uint64_t>(v);
  return n < 1 ? 1 : n;
}

static int sched_due(kh_rebuild_scheduler* s) {
  if (s->current_step >= s->next_rebuild_step) {
    s->rebuild_count += 1;
    s->next_rebuild_step = s->current_step + sched_interval(s);  // wraps as a release build
    return 1;
  }
  return 0;
}

extern "C" void kh_rebuild_scheduler_init(kh_rebuild_scheduler* s, uint64_t base_interval,
                                          double decay) {
  if (!s) return;
  s->base_interval = base_interval;
  s->decay = decay;
  s->rebuild_count = 0;
  s->next_rebuild_step = base_interval;
  s->current_step = 0;
}

extern "C" int kh_rebuild_scheduler_step(kh_rebuild_scheduler* s) {
  if (!s) return 0;
  s->current_step += 1;
  return sched_due(s);
}

extern "C" int kh_rebuild_scheduler_should_rebuild(kh_rebuild_scheduler* s, uint64_t step) {
  if (!s) return 0;
  s->current_step = step;
  return sched_due(s);
}

// ======================================================================== index / layer
extern "C" int kh_lsh_index_rebuild(kh_lsh_index* idx, const uint32_t* ids_dev, const float* w_dev,
                                    int64_t n, int64_t ldw, void* stream) {
  KH_CHECK_ARG(idx != nullptr, "null index");
  KH_CHECK_ARG(n >= 0 && ldw >= idx->h->dim, "bad n/ldw");
  int rc = kh_lsh_index_clear(idx, stream);
  if (rc != KH_OK || n == 0) return rc;
  return kh_lsh_index_insert(idx, ids_dev, w_dev, n, ldw, stream);
}

extern "C" int kh_slide_layer_rebuild_index(kh_slide_layer* l, void* stream) {
  KH_CHECK_ARG(l != nullptr, "null layer");
  uint32_t* ids = static_cast<uint32_t*>(dev_alloc(sizeof(uint32_t) * l->n));
  if (!ids) return KH_ERR_ALLOC;
  std::vector<uint32_t> h(l->n);
  for (int i = 0; i < l->n; ++i) h[i] = static_cast<uint32_t>(i);
  hipStream_t st = as_stream(stream);
  int rc = KH_OK;
  if (hipMemcpyAsync(ids, h.data(), sizeof(uint32_t) * l->n, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess) {
    set_error("rebuild upload failed");
    rc = KH_ERR_HIP;
  }
  if (rc == KH_OK) rc = kh_lsh_index_rebuild(l->index, ids, l->w, l->n, l->dim, stream);
  if (rc == KH_OK && hipStreamSynchronize(st) != hipSuccess) {
    set_error("rebuild failed");
    rc = KH_ERR_HIP;
  }
  dev_free(ids);
  return rc;
}

extern "C" int kh_slide_layer_init_optimizer(kh_slide_layer* l, int optimizer, float momentum,
                                             float beta1, float beta2, float eps) {
  KH_CHECK_ARG(l != nullptr, "null layer");
  KH_CHECK_ARG(optimizer == KH_OPT_SGD || optimizer == KH_OPT_ADAM, "bad optimizer %d", optimizer);
  l->free_opt();
  const size_t nw = static_cast<size_t>(l->n) * l->dim;
  const bool two = optimizer == KH_OPT_ADAM;
  const bool one = two || momentum > 0.0f;
  if (one) {
    l->st_w1 = static_cast<float*>(dev_alloc(sizeof(float) * nw));
    l->st_b1 = static_cast<float*>(dev_alloc(sizeof(float) * l->n));
    if (!l->st_w1 || !l->st_b1) {
      l->free_opt();
      return KH_ERR_ALLOC;
    }
  }
  if (two) {
    l->st_w2 = static_cast<float*>(dev_alloc(sizeof(float) * nw));
    l->st_b2 = static_cast<float*>(dev_alloc(sizeof(float) * l->n));
    if (!l->st_w2 || !l->st_b2) {
      l->free_opt();
      return KH_ERR_ALLOC;
    }
  }
  float* bufs[4] = {l->st_w1, l->st_w2, l->st_b1, l->st_b2};
  const size_t cnt[4] = {nw, nw, (size_t)l->n, (size_t)l->n};
  for (int i = 0; i < 4; ++i)
    if (bufs[i] && hipMemset(bufs[i], 0, sizeof(float) * cnt[i]) != hipSuccess) {
      l->free_opt();
      set_error("optimizer state clear failed");
      return KH_ERR_HIP;
    }
  l->opt = optimizer;
  l->momentum = momentum;
  l->beta1 = beta1;
  l->beta2 = beta2;
  l->eps = eps;
  return KH_OK;
}

extern "C" int kh_slide_layer_weights(const kh_slide_layer* l, float* w_host, float* bias_host) {
  KH_CHECK_ARG(l != nullptr, "null layer");
  if (w_host)
    KH_HIP(hipMemcpy(w_host, l->w, sizeof(float) * l->n * (size_t)l->dim, hipMemcpyDeviceToHost));
  if (bias_host) KH_HIP(hipMemcpy(bias_host, l->bias, sizeof(float) * l->n, hipMemcpyDeviceToHost));
  return KH_OK;
}

extern "C" int kh_slide_layer_backward(kh_slide_layer* l, const float* x_dev,
                                       const uint32_t* act_ids_dev, const int32_t* n_act_dev,
                                       const float* pre_dev, const float* act_dense_dev,
                                       const float* grad_out_dev, int64_t grad_out_len, double lr,
                                       uint64_t step, float* grad_in_dev, void* stream) {
  KH_CHECK_ARG(l != nullptr, "null layer");
  KH_CHECK_ARG(l->opt >= 0, "kh_slide_layer_init_optimizer was not called");
  KH_CHECK_ARG(x_dev && act_ids_dev && n_act_dev && pre_dev && act_dense_dev, "null argument");
  KH_CHECK_ARG(grad_out_len >= 0 && (grad_out_len == 0 || grad_out_dev), "bad grad_out");
  hipStream_t st = as_stream(stream);
  // An active list holds distinct neuron ids, so at most n entries.
  const int cap = l->n;
  WsSet* w = l->ws.get(st);
  float* go = static_cast<float*>(w->get(0, sizeof(float) * (cap + kJPad)));
  float* lg = static_cast<float*>(w->get(1, sizeof(float) * cap));
  float* post = static_cast<float*>(w->get(2, sizeof(float) * (cap + kJPad)));
  if (!go || !lg || !post) return KH_ERR_ALLOC;
  if (l->act == KH_ACT_SOFTMAX) {
    // Layer::backward recomputes apply_softmax(pre_activations) (layer.rs:147)
    hipLaunchKernelGGL(tr_softmax_kernel, dim3(1), dim3(kSmThreads), 0, st, pre_dev, act_ids_dev,
                       n_act_dev, cap, post, nullptr, (int64_t)0);
    KH_LAUNCHED();
  }
  return layer_backward_launch(l, x_dev, act_ids_dev, n_act_dev, cap, pre_dev, post,
                               act_dense_dev, grad_out_dev, grad_out_len, false, go, lg,
                               opt_args(l, lr, step), grad_in_dev, true, st);
}

// ======================================================================== network
namespace {

struct TrainBufs {
  int qs = 0, as = 0;
  uint32_t* codes = nullptr;
  uint32_t* qids = nullptr;
  uint32_t* qcnt = nullptr;
  int32_t* qlen = nullptr;
  uint32_t* aids = nullptr;
  int32_t* alen = nullptr;
  float* pre = nullptr;
  float* post = nullptr;
  float* dense = nullptr;  // [n] the layer's activations (Layer::forward's `activations`)
  float* go = nullptr;
  float* lg = nullptr;
  float* gi = nullptr;     // [dim] gradient w.r.t. the layer's input
  uint32_t* nzi = nullptr;
  float* nzv = nullptr;
  int64_t* xoff = nullptr;
};

}  // namespace

struct kh_slide_network {
  std::vector<kh_slide_layer*> layers;
  std::vector<TrainBufs> b;
  std::vector<void*> allocs;
  uint64_t step = 0;
  kh_rebuild_scheduler sched{};
  float* loss_total = nullptr;
  // The current sparse example: its nonzeros, and the same densified [in_dim].  Apart from
  // a dense example's list (b[0]), as the next one clears x_dense at these entries.
  uint32_t* x_nzi = nullptr;
  float* x_nzv = nullptr;
  int64_t* x_off = nullptr;
  float* x_dense = nullptr;
  uint32_t* labels = nullptr;
  size_t labels_cap = 0;
  kh::StreamWs rows_ws;      // net_predict_rows' buffers, a slot of each stream
  std::mutex rows_mu;        // one prediction is enqueued at a time: host threads may share a stream
  int in_dim = 0, out_dim = 0;
  template <typename T>
  T* alloc(size_t n, bool zero = false) {
    void* p = dev_alloc(sizeof(T) * (n ? n : 1));
    if (!p) return nullptr;
    allocs.push_back(p);
    if (zero && hipMemset(p, 0, sizeof(T) * (n ? n : 1)) != hipSuccess) return nullptr;
    return static_cast<T*>(p);
  }
};

extern "C" int kh_slide_network_destroy(kh_slide_network* n) {
  if (!n) return KH_OK;
  for (void* p : n->allocs) dev_free(p);
  dev_free(n->labels);
  delete n;
  return KH_OK;
}

extern "C" int kh_slide_network_create(kh_slide_layer* const* layers, int n_layers, int optimizer,
                                       float momentum, float beta1, float beta2, float eps,
                                       uint64_t rebuild_base, double rebuild_decay,
                                       kh_slide_network** out) {
  KH_CHECK_ARG(out && layers && n_layers > 0, "null argument / no layers");
  *out = nullptr;
  for (int i = 0; i < n_layers; ++i) {
    KH_CHECK_ARG(layers[i] != nullptr, "null layer %d", i);
    KH_CHECK_ARG(i == 0 || layers[i]->dim == layers[i - 1]->n,
                 "layer %d input_dim %d != layer %d num_neurons %d", i, layers[i]->dim, i - 1,
                 layers[i - 1]->n);
    const kh_lsh_index* idx = layers[i]->index;
    KH_CHECK_ARG(layers[i]->sampling != KH_SAMPLING_TOPK || idx->L * idx->cap + 1 <= 8193,
                 "top-k sampling supports num_tables * bucket_capacity <= 8192");
  }
  auto* net = new kh_slide_network();
  net->layers.assign(layers, layers + n_layers);
  net->in_dim = layers[0]->dim;
  net->out_dim = layers[n_layers - 1]->n;
  kh_rebuild_scheduler_init(&net->sched, rebuild_base, rebuild_decay);
  int rc = KH_OK;
  for (int i = 0; i < n_layers && rc == KH_OK; ++i)
    rc = kh_slide_layer_init_optimizer(layers[i], optimizer, momentum, beta1, beta2, eps);
  net->b.resize(n_layers);
  for (int i = 0; i < n_layers && rc == KH_OK; ++i) {
    const kh_slide_layer* l = layers[i];
    TrainBufs& t = net->b[i];
    t.qs = l->index->L * l->index->cap;
    t.as = std::max(t.qs, l->n);
    t.codes = net->alloc<uint32_t>(l->index->L);
    t.qids = net->alloc<uint32_t>(t.qs);
    t.qcnt = net->alloc<uint32_t>(t.qs);
    t.qlen = net->alloc<int32_t>(1, true);
    t.aids = net->alloc<uint32_t>(t.as, true);
    t.alen = net->alloc<int32_t>(1, true);
    t.pre = net->alloc<float>(t.as);
    t.post = net->alloc<float>(t.as + kJPad);
    t.dense = net->alloc<float>(l->n, true);
    t.go = net->alloc<float>(t.as + kJPad);
    t.lg = net->alloc<float>(t.as);
    t.gi = net->alloc<float>(l->dim);
    t.nzi = net->alloc<uint32_t>(l->dim);
    t.nzv = net->alloc<float>(l->dim);
    t.xoff = net->alloc<int64_t>(2, true);
    if (!t.codes || !t.qids || !t.qcnt || !t.qlen || !t.aids || !t.alen || !t.pre || !t.post ||
        !t.dense || !t.go || !t.lg || !t.gi || !t.nzi || !t.nzv || !t.xoff)
      rc = KH_ERR_ALLOC;
  }
  if (rc == KH_OK) {
    net->loss_total = net->alloc<float>(1, true);
    net->x_nzi = net->alloc<uint32_t>(net->in_dim);
    net->x_nzv = net->alloc<float>(net->in_dim);
    net->x_off = net->alloc<int64_t>(2, true);
    net->x_dense = net->alloc<float>(net->in_dim, true);
    if (!net->loss_total || !net->x_nzi || !net->x_nzv || !net->x_off || !net->x_dense) rc = KH_ERR_ALLOC;
  }
  if (rc != KH_OK) {
    kh_slide_network_destroy(net);
    return rc;
  }
  *out = net;
  return KH_OK;
}

// Stage example e of a CSR batch as layer 0's input (to_dense semantics).
static int net_stage_sparse(kh_slide_network* net, const int64_t* xoff, const uint32_t* xidx,
                            const float* xval, int64_t e, hipStream_t st) {
  hipLaunchKernelGGL(tr_stage_csr_kernel, dim3(1), dim3(1024), 0, st, xoff, xidx, xval, e,
                     net->in_dim, (int64_t)0, net->x_nzi, net->x_nzv, net->x_off, net->x_dense);
  KH_LAUNCHED();
  return KH_OK;
}

// Host check of a CSR batch: offsets nondecreasing, at most kTrMaxNnz stored
// entries per example (reads the offsets back; synchronous).
static int net_check_csr(const int64_t* xoff, int64_t batch, hipStream_t st) {
  std::vector<int64_t> off(batch + 1);
  KH_HIP(hipMemcpyAsync(off.data(), xoff, sizeof(int64_t) * (batch + 1), hipMemcpyDeviceToHost, st));
  KH_HIP(hipStreamSynchronize(st));
  for (int64_t e = 0; e < batch; ++e)
    KH_CHECK_ARG(off[e + 1] >= off[e] && off[e + 1] - off[e] <= kTrMaxNnz,
                 "example %lld: offsets must be nondecreasing with at most %d entries", (long long)e,
                 kTrMaxNnz);
  return KH_OK;
}

// Network::forward for one example (net.rs:62-78), layer by layer: nonzeros of
// the input, hash, query, sampling in the sampler's order (clearing the
// previous example's entries of the dense activations), neuron sums, softmax.
// x == nullptr: layer 0's input was staged from a sparse example.
static int net_forward_one(kh_slide_network* net, const float* x, hipStream_t st) {
  const float* in = x;
  for (size_t i = 0; i < net->layers.size(); ++i) {
    kh_slide_layer* l = net->layers[i];
    TrainBufs& t = net->b[i];
    // short dense inputs need no list of nonzeros: the per-row hash and the tile
    // kernel read them as they are (128 -> 8191 neurons, 4470
    // active: hash 4.2 and sums 7.1 us, against 4.6 + 5.8 + 21 with the list)
    const bool tile = in && hash_dense_rows(l->index->h) && neuron_tile_ok(l);
    const uint32_t* nzi = in ? t.nzi : net->x_nzi;
    const float* nzv = in ? t.nzv : net->x_nzv;
    const int64_t* xoff = in ? t.xoff : net->x_off;
    if (in && !tile) {
      hipLaunchKernelGGL(tr_stage_nz_kernel, dim3(1), dim3(1024), 0, st, in, l->dim, (int64_t)0, (int64_t)0,
                         t.nzi, t.nzv, t.xoff);
      KH_LAUNCHED();
    }
    int rc = tile ? hash_dense_launch(l->index->h, in, l->dim, 1, t.codes, st)
                  : hash_sparse_launch(l->index->h, xoff, nzi, nzv, 1, t.codes, st);
    if (rc != KH_OK) return rc;
    const int qs = query_stride(l->index);
    rc = query_launch(l->index, t.codes, 1, t.qids, t.qcnt, qs, t.qlen, st);
    if (rc != KH_OK) return rc;
    // the sampler's order only where a sum runs over the list: a softmax, or the
    // grad_input that every layer but the first computes
    rc = select_launch(l, t.qids, t.qcnt, t.qlen, qs, 1, t.aids, t.as, t.alen,
                       l->act == KH_ACT_SOFTMAX || i > 0, t.dense, st);
    if (rc != KH_OK) return rc;
    if (tile) {
      rc = neuron_tile_launch(l, in, 1, t.aids, t.as, t.alen, t.pre, t.post, t.dense, 0, st);
      if (rc != KH_OK) return rc;
    } else {
      const unsigned nb = static_cast<unsigned>(std::min(ceil_div(t.as, kTrThreads / 64), 4096));
      hipLaunchKernelGGL(tr_neuron_wave_kernel, dim3(nb), dim3(kTrThreads), 0, st, l->w, l->bias, l->dim, nzi, nzv,
                         xoff, t.aids, t.alen, t.as, l->act, t.pre, t.post, t.dense);
      KH_LAUNCHED();
    }
    if (l->act == KH_ACT_SOFTMAX) {
      hipLaunchKernelGGL(tr_softmax_kernel, dim3(1), dim3(kSmThreads), 0, st, t.pre, t.aids, t.alen,
                         t.as, t.post, t.dense, (int64_t)0);
      KH_LAUNCHED();
    }
    in = t.dense;
  }
  return KH_OK;
}

static int net_setup_attrs() {
  static int rc = [] {
    const size_t lds = (sizeof(uint32_t) + sizeof(float)) * kTrLdsNz;
    for (const void* k : {reinterpret_cast<const void*>(&tr_neuron_kernel<false>),
                          reinterpret_cast<const void*>(&tr_neuron_kernel<true>)})
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
        return static_cast<int>(KH_ERR_HIP);
    return static_cast<int>(KH_OK);
  }();
  if (rc != KH_OK) set_error("hipFuncSetAttribute failed");
  return rc;
}

// Network::train_step over dense rows (x_dev) or CSR rows (xoff != nullptr).
static int net_train_step(kh_slide_network* net, const float* x_dev, const int64_t* xoff,
                          const uint32_t* xidx, const float* xval, int64_t batch,
                          const int64_t* label_off_host, const uint32_t* labels_host, double lr,
                          float* loss_out, void* stream) {
  KH_CHECK_ARG(net && loss_out, "null argument");
  KH_CHECK_ARG(batch >= 0, "bad batch");
  *loss_out = 0.0f;
  if (batch == 0) return KH_OK;  // net.rs:82-84: nothing changes
  KH_CHECK_ARG((x_dev || xoff) && label_off_host, "null input");
  KH_CHECK_ARG(label_off_host[0] == 0, "label offsets must start at 0");
  for (int64_t e = 0; e < batch; ++e)
    KH_CHECK_ARG(label_off_host[e + 1] >= label_off_host[e] &&
                     label_off_host[e + 1] - label_off_host[e] <= kTrMaxLabels,
                 "example %lld: label offsets must be nondecreasing with at most %d labels",
                 (long long)e, kTrMaxLabels);
  const int64_t n_labels = label_off_host[batch];
  KH_CHECK_ARG(n_labels == 0 || labels_host, "null labels");
  int rc = KH_OK;
  hipStream_t st = as_stream(stream);
  if (xoff) {
    rc = net_check_csr(xoff, batch, st);
    if (rc != KH_OK) return rc;
  }
  if (static_cast<size_t>(n_labels) > net->labels_cap) {
    KH_HIP(hipStreamSynchronize(st));
    dev_free(net->labels);
    net->labels_cap = std::max<size_t>(n_labels, 2 * net->labels_cap);
    net->labels = static_cast<uint32_t*>(dev_alloc(sizeof(uint32_t) * net->labels_cap));
    if (!net->labels) {
      net->labels_cap = 0;
      return KH_ERR_ALLOC;
    }
  }
  if (n_labels)
    KH_HIP(hipMemcpyAsync(net->labels, labels_host, sizeof(uint32_t) * n_labels,
                          hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(fill_f32_kernel<>, dim3(1), dim3(64), 0, st, net->loss_total, (int64_t)1, 0.0f);
  KH_LAUNCHED();
  const int nl_layers = static_cast<int>(net->layers.size());
  std::vector<OptArgs> oa(nl_layers);
  for (int i = 0; i < nl_layers; ++i) oa[i] = opt_args(net->layers[i], lr, net->step);
  for (int64_t e = 0; e < batch; ++e) {
    const float* x = xoff ? net->x_dense : x_dev + e * static_cast<int64_t>(net->in_dim);
    if (xoff) {
      rc = net_stage_sparse(net, xoff, xidx, xval, e, st);
      if (rc != KH_OK) return rc;
    }
    rc = net_forward_one(net, xoff ? nullptr : x, st);
    if (rc != KH_OK) return rc;
    const int last = nl_layers - 1;
    kh_slide_layer* L = net->layers[last];
    TrainBufs& T = net->b[last];
    const int nl = static_cast<int>(label_off_host[e + 1] - label_off_host[e]);
    hipLaunchKernelGGL(tr_loss_grad_kernel, dim3(1), dim3(kLossThreads), 0, st, T.pre, T.post, T.aids,
                       T.alen, T.as, L->act, T.dense, net->labels + label_off_host[e], nl, T.go,
                       T.lg, net->loss_total);
    KH_LAUNCHED();
    // Network::backward (net.rs:122-146): last layer down to the first
    for (int i = last; i >= 0; --i) {
      kh_slide_layer* l = net->layers[i];
      TrainBufs& t = net->b[i];
      const float* in = i == 0 ? x : net->b[i - 1].dense;
      const float* grad_out = i == last ? nullptr : net->b[i + 1].gi;
      // the first layer's grad_input is not used by anything (net.rs:139-144)
      float* gi = i == 0 ? nullptr : t.gi;
      rc = layer_backward_launch(l, in, t.aids, t.alen, t.as, t.pre, t.post, t.dense, grad_out,
                                 l->n, i == last, t.go, t.lg, oa[i], gi, false, st);
      if (rc != KH_OK) return rc;
    }
  }
  for (kh_slide_layer* l : net->layers) {
    rc = wtn_refresh(l, st);
    if (rc != KH_OK) return rc;
  }
  float total = 0.0f;
  KH_HIP(hipMemcpyAsync(&total, net->loss_total, sizeof(float), hipMemcpyDeviceToHost, st));
  KH_HIP(hipStreamSynchronize(st));
  net->step += 1;
  if (kh_rebuild_scheduler_should_rebuild(&net->sched, net->step)) {
    for (kh_slide_layer* l : net->layers) {
      rc = kh_slide_layer_rebuild_index(l, stream);
      if (rc != KH_OK) return rc;
    }
  }
  *loss_out = total / static_cast<float>(batch);
  return KH_OK;
}

extern "C" int kh_slide_network_train_step(kh_slide_network* net, const float* x_dev, int64_t batch,
                                           const int64_t* label_off_host,
                                           const uint32_t* labels_host, double lr, float* loss_out,
                                           void* stream) {
  KH_CHECK_ARG(batch == 0 || x_dev, "null input");
  return net_train_step(net, x_dev, nullptr, nullptr, nullptr, batch, label_off_host, labels_host,
                        lr, loss_out, stream);
}

extern "C" int kh_slide_network_train_step_sparse(kh_slide_network* net, const int64_t* xoff_dev,
                                                  const uint32_t* xidx_dev, const float* xval_dev,
                                                  int64_t batch, const int64_t* label_off_host,
                                                  const uint32_t* labels_host, double lr,
                                                  float* loss_out, void* stream) {
  KH_CHECK_ARG(batch == 0 || xoff_dev, "null input");
  return net_train_step(net, nullptr, xoff_dev, xidx_dev, xval_dev, batch, label_off_host,
                        labels_host, lr, loss_out, stream);
}

// While it lives, this thread may allocate beside a capture (allocations are not captured).
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Network::forward for a batch, a row per example: the kernels of
// net_forward_one over `rows` examples at a time, so a batch costs one chain of
// launches instead of one per example (784 -> 1024 -> 32, batch 128: 71 us,
// against 17.1 ms for 128 chains, each bound by its launches' latency).  Ternary families whose
// signs fit the per-row LDS kernel hash the dense rows; the others hash the
// staged lists, as net_forward_one does (the codes are the same).  The rows
// taken at a time keep the scratch within kRowsWs bytes (at least one row).  The
// scratch is the stream's own, as a prediction writes nothing else and may run
// beside others; it grows under stream capture too.
constexpr size_t kRowsWs = (size_t)256 << 20;
static int net_predict_rows(kh_slide_network* net, const float* x_dev, const int64_t* xoff,
                            const uint32_t* xidx, const float* xval, int64_t batch, float* out_dev,
                            hipStream_t st) {
  auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t nl = net->layers.size();
  // per-row entries of each buffer: the largest layer's (dense activations
  // between layers are kept apart: two alternate)
  size_t mL = 0, mqs = 0, mas = 0, mnz = 0, mdense = 0;
  std::vector<int> qs(nl), as(nl);
  for (size_t i = 0; i < nl; ++i) {
    const kh_slide_layer* l = net->layers[i];
    qs[i] = query_stride(l->index);
    as[i] = std::max(qs[i], l->n);
    mL = std::max(mL, (size_t)l->index->L);
    mqs = std::max(mqs, (size_t)qs[i]);
    mas = std::max(mas, (size_t)as[i]);
    mnz = std::max(mnz, (size_t)(i == 0 && xoff ? std::min(l->dim, kTrMaxNnz) : l->dim));
    if (i + 1 < nl) mdense = std::max(mdense, (size_t)l->n);
  }
  const size_t per_row = sizeof(int64_t) * 2 + 4 * (mL + 2 * mqs + 3 * mas + 2 * mnz + 2 * mdense + 2);
  constexpr int kBufs = 13;
  size_t sizes[kBufs];
  int64_t rows = std::min<int64_t>({batch, std::max<int64_t>(1, (int64_t)(kRowsWs / per_row)), 65535});
  char* base = nullptr;
  for (;; rows /= 2) {   // fewer rows at a time where memory is short
    const size_t R = (size_t)rows;
    const size_t need[kBufs] = {R * 16, 4 * R * mL, 4 * R * mqs, 4 * R * mqs, 4 * R, 4 * R * mas, 4 * R, 4 * R * mas,
                                4 * R * mas, 4 * R * mnz, 4 * R * mnz, 4 * R * mdense, 4 * R * mdense};
    size_t total = 0;
    for (int i = 0; i < kBufs; ++i) total += sizes[i] = pad(need[i]);
    RelaxedCapture relaxed;
    base = static_cast<char*>(net->rows_ws.get(st)->get(0, total));
    if (base) break;
    if (rows == 1) return KH_ERR_ALLOC;
    (void)hipGetLastError();
  }
  char* buf[kBufs];
  for (int i = 0; i < kBufs; ++i) {
    buf[i] = base;
    base += sizes[i];
  }
  auto* nzoff = reinterpret_cast<int64_t*>(buf[0]);
  auto* codes = reinterpret_cast<uint32_t*>(buf[1]);
  auto* qids = reinterpret_cast<uint32_t*>(buf[2]);
  auto* qcnt = reinterpret_cast<uint32_t*>(buf[3]);
  auto* qlen = reinterpret_cast<int32_t*>(buf[4]);
  auto* aids = reinterpret_cast<uint32_t*>(buf[5]);
  auto* alen = reinterpret_cast<int32_t*>(buf[6]);
  auto* pre = reinterpret_cast<float*>(buf[7]);
  auto* post = reinterpret_cast<float*>(buf[8]);
  auto* nzi = reinterpret_cast<uint32_t*>(buf[9]);
  auto* nzv = reinterpret_cast<float*>(buf[10]);
  float* hidden[2] = {reinterpret_cast<float*>(buf[11]), reinterpret_cast<float*>(buf[12])};
  for (int64_t e0 = 0; e0 < batch; e0 += rows) {
    const int64_t nr = std::min(rows, batch - e0);
    const float* in = xoff ? nullptr : x_dev + e0 * net->in_dim;
    for (size_t i = 0; i < nl; ++i) {
      const kh_slide_layer* l = net->layers[i];
      const kh_hash_family* h = l->index->h;
      const int64_t stride = in ? l->dim : std::min(l->dim, kTrMaxNnz);
      if (in)
        hipLaunchKernelGGL(tr_stage_nz_kernel, dim3((unsigned)nr), dim3(1024), 0, st, in, l->dim,
                           (int64_t)l->dim, stride, nzi, nzv, nzoff);
      else
        hipLaunchKernelGGL(tr_stage_csr_kernel, dim3((unsigned)nr), dim3(1024), 0, st, xoff, xidx, xval, e0,
                           l->dim, stride, nzi, nzv, nzoff, (float*)nullptr);
      KH_LAUNCHED();
      int rc = in && hash_dense_rows(h)
                   ? hash_dense_launch(h, in, l->dim, nr, codes, st)
                   : hash_sparse_launch(h, nzoff, nzi, nzv, nr, codes, st, 2);
      if (rc != KH_OK) return rc;
      rc = query_launch(l->index, codes, nr, qids, qcnt, qs[i], qlen, st);
      if (rc != KH_OK) return rc;
      // Only a softmax's sum depends on the list's order; elsewhere ascending ids,
      // whose weights in a row of the transposed copy lie close together.
      rc = select_launch(l, qids, qcnt, qlen, qs[i], nr, aids, as[i], alen, l->act == KH_ACT_SOFTMAX, nullptr, st);
      if (rc != KH_OK) return rc;
      float* dense = i + 1 < nl ? hidden[i & 1] : out_dev + e0 * net->out_dim;
      hipLaunchKernelGGL(fill_f32_kernel<>, dim3((unsigned)ceil_div(nr * l->n, 256)), dim3(256), 0, st, dense,
                         nr * l->n, 0.0f);
      KH_LAUNCHED();
      // enough blocks for the chip; a row's blocks past its list leave at once
      const int nb = std::min(ceil_div(as[i], kTrThreads), std::max(1, 4096 / (int)nr));
      const int lds_nz = std::min<int>(kTrLdsNz, entries_padded((int)stride));
      const size_t lds = (sizeof(uint32_t) + sizeof(float)) * lds_nz;
      const dim3 g((unsigned)nb, (unsigned)nr);
      if (l->wtn)
        hipLaunchKernelGGL(tr_neuron_kernel<true>, g, dim3(kTrThreads), lds, st, l->wtn, l->bias, l->dim, l->n, lds_nz, nzi, nzv,
                           nzoff, aids, alen, as[i], l->act, pre, post, dense, (int64_t)l->n);
      else
        hipLaunchKernelGGL(tr_neuron_kernel<false>, g, dim3(kTrThreads), lds, st, l->w, l->bias, l->dim, l->dim, lds_nz, nzi, nzv,
                           nzoff, aids, alen, as[i], l->act, pre, post, dense, (int64_t)l->n);
      KH_LAUNCHED();
      if (l->act == KH_ACT_SOFTMAX) {
        hipLaunchKernelGGL(tr_softmax_kernel, dim3((unsigned)nr), dim3(kSmThreads), 0, st, pre, aids, alen, as[i],
                           post, dense, (int64_t)l->n);
        KH_LAUNCHED();
      }
      in = dense;
    }
  }
  return KH_OK;
}

static int net_predict(kh_slide_network* net, const float* x_dev, const int64_t* xoff,
                       const uint32_t* xidx, const float* xval, int64_t batch, float* out_dev,
                       void* stream) {
  KH_CHECK_ARG(net != nullptr, "null network");
  KH_CHECK_ARG(batch >= 0, "bad batch");
  if (batch == 0) return KH_OK;
  KH_CHECK_ARG((x_dev || xoff) && out_dev, "null argument");
  int rc = net_setup_attrs();
  if (rc != KH_OK) return rc;
  hipStream_t st = as_stream(stream);
  if (xoff) {
    rc = net_check_csr(xoff, batch, st);
    if (rc != KH_OK) return rc;
  }
  std::lock_guard<std::mutex> g(net->rows_mu);
  return net_predict_rows(net, x_dev, xoff, xidx, xval, batch, out_dev, st);
}

extern "C" int kh_slide_network_predict(kh_slide_network* net, const float* x_dev, int64_t batch,
                                        float* out_dev, void* stream) {
  return net_predict(net, x_dev, nullptr, nullptr, nullptr, batch, out_dev, stream);
}

extern "C" int kh_slide_network_predict_sparse(kh_slide_network* net, const int64_t* xoff_dev,
                                               const uint32_t* xidx_dev, const float* xval_dev,
                                               int64_t batch, float* out_dev, void* stream) {
  return net_predict(net, nullptr, xoff_dev, xidx_dev, xval_dev, batch, out_dev, stream);
}

extern "C" int kh_slide_network_state(const kh_slide_network* net, uint64_t* step,
                                      kh_rebuild_scheduler* scheduler) {
  KH_CHECK_ARG(net != nullptr, "null network");
  if (step) *step = net->step;
  if (scheduler) *scheduler = net->sched;
  return KH_OK;
}
