// slide.hip -- SLIDE sparse layer forward on the GPU (gfx950).
//
// Replaces Layer::forward (crates/klearu-core/src/network/layer.rs:65-120) with
// Neuron::forward / forward_sparse (network/neuron.rs:47-68), the sampling
// strategies (sampling/{vanilla,topk,threshold}.rs) and the activations
// (layer.rs:250-308); plus a dense layer over sparse inputs (every neuron,
// Neuron::forward_sparse) for the hidden layer of the extreme-classification net.
//
// Per batch: hash (lsh.hip) -> query (unique ids + hit counts, ascending) ->
// select_kernel (sampling, empty -> all neurons, ids < n) -> neuron_kernel
// (one block per sample; each thread replays the reference's sequential f32
// sum for one active neuron over the sample's nonzero inputs, then the
// activation; softmax reduces over the block) -> CSR.
//
// Skipping zero inputs leaves a sequential sum unchanged (adding +-0 to a
// nonzero partial sum returns it; a zero partial sum only changes the sign of
// zero), so pre-activations are bit-identical to the reference's dense loop.
#include <algorithm>
#include <mutex>
#include <vector>

#include "gather.hpp"
#include "entry_sum.hpp"
#include "slide_internal.hpp"

namespace kh {

constexpr int kSlideThreads = 256;
constexpr int kMaxCountBins = 8193;

// Top-k sampling in the sampler's own order (count descending, then id, as
// TopKSampling::select sorts, sampling/topk.rs:19-34): a stable counting sort
// of the ascending candidates.  hist[c] becomes the number of candidates with
// a count above c; wave 0 then walks the candidates in id order and places
// each after the earlier ones of its count.  Returns min(m, top_k), the
// sampler's pick count; picks with ids >= num_neurons are dropped in order.
__device__ int select_topk_count_order(const uint32_t* __restrict__ ids,
                                       const uint32_t* __restrict__ cnt, int m, int top_k,
                                       int num_neurons, int nbins, unsigned* hist, int* wsum,
                                       int* s_total, uint32_t* __restrict__ out, int* n_kept) {
  for (int i = threadIdx.x; i < nbins; i += blockDim.x) hist[i] = 0u;
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += blockDim.x) atomicAdd(&hist[cnt[i]], 1u);
  __syncthreads();
  // exclusive suffix sums: thread t owns a run of bins, thread 0 the highest
  const int seg = (nbins + (int)blockDim.x - 1) / (int)blockDim.x;
  const int hi = nbins - 1 - (int)threadIdx.x * seg;
  const int lo = max(hi - seg + 1, 0);
  int run = 0;
  for (int c = hi; c >= lo; --c) run += (int)hist[c];
  int above = block_excl_scan(run, wsum, s_total);
  for (int c = hi; c >= lo; --c) {
    const int h = (int)hist[c];
    hist[c] = (unsigned)above;
    above += h;
  }
  __syncthreads();
  const int take = min(m, top_k);
  if ((threadIdx.x >> 6) == 0) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    for (int c0 = 0; c0 < m; c0 += 64) {
      const int i = c0 + lane;
      const int c = i < m ? (int)cnt[i] : -1;
      uint64_t pend = __ballot(i < m);
      while (pend) {
        const int leader = __ffsll((unsigned long long)pend) - 1;
        const int cl = __shfl(c, leader);
        const uint64_t same = __ballot(c == cl);
        const int base = (int)hist[cl];
        if (c == cl) {
          const int pos = base + __popcll(same & below);
          if (pos < take) out[pos] = ids[i];
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == leader) hist[cl] = (unsigned)(base + __popcll(same));
        __builtin_amdgcn_wave_barrier();
        pend &= ~same;
      }
    }
  }
  __syncthreads();
  // drop ids >= num_neurons, keeping the order (layer.rs:87)
  int base = 0;
  for (int c0 = 0; c0 < take; c0 += blockDim.x) {
    const int i = c0 + threadIdx.x;
    const uint32_t id = i < take ? out[i] : 0u;
    const int keep = i < take && id < (uint32_t)num_neurons;
    const int pos = block_excl_scan(keep, wsum, s_total) + base;
    if (keep) out[pos] = id;
    base += *s_total;
    __syncthreads();
  }
  *n_kept = base;
  return take;
}

// clear_dense (training): the row's dense activation vector [num_neurons];
// the entries of the previous active list (aids/alen still hold it) are
// zeroed before the new list is written.  count_order: top-k picks in the
// sampler's order instead of ascending ids.  ids_below: every candidate id is
// below num_neurons, so a selection of all candidates is a copy of the list
// (one row of 4470 candidates: 3.4 us; 15 when each thread walked its own run
// of them twice, with 256 threads).
constexpr int kSelectThreads = 1024;       // rows up to kSelectFewRows; kSlideThreads beyond
constexpr int64_t kSelectFewRows = 256;
__global__ __launch_bounds__(kSelectThreads) void select_kernel(
    const uint32_t* __restrict__ qids, const uint32_t* __restrict__ qcnt,
    const int32_t* __restrict__ qlen, int qstride, int sampling, int top_k, int threshold,
    int num_neurons, int nbins, uint32_t* __restrict__ aids, int astride,
    int32_t* __restrict__ alen, int count_order, float* __restrict__ clear_dense, int fallback,
    int ids_below) {
  extern __shared__ unsigned hist[];
  __shared__ int wsum[kSelectThreads / 64];
  __shared__ int s_total;
  __shared__ int s_cstar, s_take, s_best_id;
  const int64_t row = blockIdx.x;
  const uint32_t* ids = qids + row * (int64_t)qstride;
  const uint32_t* cnt = qcnt + row * (int64_t)qstride;
  uint32_t* out = aids + row * (int64_t)astride;
  const int m = qlen[row];
  if (clear_dense) {
    float* dn = clear_dense + row * (int64_t)num_neurons;
    const int old = alen[row];
    constexpr int U = 4;
    for (int a = threadIdx.x; a < old; a += blockDim.x * U) {
      uint32_t id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) id[u] = out[min(a + u * (int)blockDim.x, old - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) dn[id[u]] = 0.0f;
    }
    __syncthreads();
  }
  int cstar = 0, take_eq = 0;  // topk: take count > cstar, plus take_eq of count == cstar
  int mode = sampling;
  if (sampling == KH_SAMPLING_TOPK && count_order) {
    int n_kept = 0;
    const int n_pre = select_topk_count_order(ids, cnt, m, top_k, num_neurons, nbins, hist, wsum,
                                              &s_total, out, &n_kept);
    int n_sel = n_kept;
    if (n_pre == 0 && fallback) {
      for (int i = threadIdx.x; i < num_neurons; i += blockDim.x) out[i] = (uint32_t)i;
      n_sel = num_neurons;
    }
    if (threadIdx.x == 0) alen[row] = n_sel;
    return;
  }
  if (sampling == KH_SAMPLING_TOPK) {
    if (m <= top_k) {
      mode = KH_SAMPLING_VANILLA;
    } else {
      for (int i = threadIdx.x; i < nbins; i += blockDim.x) hist[i] = 0u;
      __syncthreads();
      for (int i = threadIdx.x; i < m; i += blockDim.x) atomicAdd(&hist[cnt[i]], 1u);
      __syncthreads();
      // Find the count c* where the number of candidates with count >= c*
      // first reaches top_k.  Thread t owns a run of bins, thread 0 the
      // highest; an exclusive scan gives each run the number of candidates
      // above it, and the run holding the crossing walks its bins downwards.
      if (threadIdx.x == 0) {
        s_cstar = 0;
        s_take = top_k;
      }
      const int seg = (nbins + (int)blockDim.x - 1) / (int)blockDim.x;
      const int hi = nbins - 1 - (int)threadIdx.x * seg;
      const int lo = max(hi - seg + 1, 0);
      int run = 0;
      for (int c = hi; c >= lo; --c) run += (int)hist[c];
      const int above = block_excl_scan(run, wsum, &s_total);
      if (hi >= 0 && above < top_k && above + run >= top_k) {
        int a = above, c = hi;
        for (; c > lo; --c) {
          if (a + (int)hist[c] >= top_k) break;
          a += (int)hist[c];
        }
        s_cstar = c;
        s_take = top_k - a;
      }
      __syncthreads();
      cstar = s_cstar;
      take_eq = s_take;
    }
  }
  // n_pre counts the sampler's picks before ids >= num_neurons are dropped:
  // the all-neurons fallback (layer.rs:82-84) runs before that filter (:87).
  int n_sel = 0, n_pre = 0;
  if (mode == KH_SAMPLING_VANILLA && ids_below) {
    constexpr int U = 4;
    for (int i = threadIdx.x; i < m; i += blockDim.x * U) {
      uint32_t id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) id[u] = ids[min(i + u * (int)blockDim.x, m - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) out[min(i + u * (int)blockDim.x, m - 1)] = id[u];
    }
    n_sel = n_pre = m;
  } else if (mode == KH_SAMPLING_THRESHOLD) {
    int base = 0, passed = 0;
    for (int c0 = 0; c0 < m; c0 += blockDim.x) {
      const int i = c0 + threadIdx.x;
      const int sel = (i < m && cnt[i] >= (uint32_t)threshold) ? 1 : 0;
      const int id = i < m ? (int)ids[i] : 0;
      const int keep = sel && (uint32_t)id < (uint32_t)num_neurons;
      block_excl_scan(sel, wsum, &s_total);
      passed += s_total;
      const int pos = block_excl_scan(keep, wsum, &s_total) + base;
      if (keep) out[pos] = (uint32_t)id;
      base += s_total;
    }
    n_sel = base;
    n_pre = passed;
    if (m > 0 && passed == 0) {
      // threshold.rs:37-42: the single best candidate (highest count, then
      // lowest id; ids are ascending, so the first maximum).
      if (threadIdx.x == 0) {
        uint32_t bc = 0, bi = ids[0];
        for (int i = 0; i < m; ++i)
          if (cnt[i] > bc || i == 0) {
            bc = cnt[i];
            bi = ids[i];
          }
        s_best_id = (int)bi;
      }
      __syncthreads();
      n_pre = 1;
      n_sel = 0;
      if ((uint32_t)s_best_id < (uint32_t)num_neurons) {
        if (threadIdx.x == 0) out[0] = (uint32_t)s_best_id;
        n_sel = 1;
      }
    }
  } else {
    // Thread t owns the candidates [t*R, t*R + R) in order, so one block scan
    // per quantity gives every output position: the rank among the count ==
    // c* candidates (top-k), then the position among the kept ones.
    // No pick at all (no candidates, or top-k of 0) writes nothing: the
    // all-neurons fallback below then owns the output.
    const bool topk = mode == KH_SAMPLING_TOPK;
    n_pre = topk ? min(m, top_k) : m;
    const int R = n_pre > 0 ? (m + (int)blockDim.x - 1) / (int)blockDim.x : 0;
    const int i0 = min((int)threadIdx.x * R, m), i1 = min(i0 + R, m);
    int eq_base = 0;
    if (topk) {
      int n_eq = 0;
      for (int i = i0; i < i1; ++i) n_eq += (int)cnt[i] == cstar ? 1 : 0;
      eq_base = block_excl_scan(n_eq, wsum, &s_total);
    }
    int n_keep = 0;
    for (int i = i0, r = eq_base; i < i1; ++i) {
      bool sel = true;
      if (topk) {
        const int c = (int)cnt[i];
        sel = c > cstar || (c == cstar && r < take_eq);
        r += c == cstar ? 1 : 0;
      }
      n_keep += sel && ids[i] < (uint32_t)num_neurons ? 1 : 0;
    }
    int pos = block_excl_scan(n_keep, wsum, &s_total);
    n_sel = s_total;
    for (int i = i0, r = eq_base; i < i1; ++i) {
      bool sel = true;
      if (topk) {
        const int c = (int)cnt[i];
        sel = c > cstar || (c == cstar && r < take_eq);
        r += c == cstar ? 1 : 0;
      }
      const uint32_t id = ids[i];
      if (sel && id < (uint32_t)num_neurons) out[pos++] = id;
    }
  }
  // empty selection -> every neuron (layer.rs:82-84)
  if (n_pre == 0 && fallback) {
    for (int i = threadIdx.x; i < num_neurons; i += blockDim.x) out[i] = (uint32_t)i;
    n_sel = num_neurons;
  }
  if (threadIdx.x == 0) alen[row] = n_sel;
}

// One block per sample (several per sample without softmax: blockIdx.y takes
// every gridDim.y-th block of active ids).  x is either dense [batch][dim]
// (zeros skipped) or CSR.  TRANS: W is the transposed copy [dim][nn].
// fb_n > 0 (Vanilla sampling read straight from the query, every id below the
// layer's fb_n neurons): a sample whose candidate list is empty takes all fb_n
// neurons (layer.rs:82-84), whose ids the blocks write into its aids row; the
// row lengths the outputs use go to alen_out (vanilla_len decides).
__device__ __forceinline__ int vanilla_len(const int32_t* alen, int64_t row, int fb_n, bool& all) {
  const int n = alen[row];
  all = fb_n > 0 && n == 0;
  return all ? fb_n : n;
}
// Where a forward's CSR rows go.  A block sums the lengths before its row itself (up to
// kCsrPackMax rows; longer batches and off == nullptr leave rows in pre / post for a
// packing launch), so entries are written once, in place; a row that does not fit
// below `capacity` is worked out in pre / post and its head copied, the caller then
// reports the overflow.  The packing launch took 4 us (128 rows of 1000) and 18 us
// (256 rows of 6400) besides the second pass over the values.
struct CsrOut {
  int64_t* off;
  uint32_t* ids;
  float *pre, *act;
  int64_t batch, capacity;
};
struct CsrRow {
  int64_t o;       // the row's first entry
  bool direct;     // it fits
  float *pre, *act;
};
// Before a barrier: this wave's part of the lengths before `row`.
__device__ __forceinline__ void csr_part(const CsrOut& co, const int32_t* alen, int64_t row, int fb_n, long long* part) {
  if (!co.off) return;
  long long s = 0;
  for (int64_t r = threadIdx.x; r < row; r += blockDim.x) {
    bool all;
    s += vanilla_len(alen, r, fb_n, all);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
}
// After it.
__device__ __forceinline__ CsrRow csr_row(const CsrOut& co, int64_t row, int n, const long long* part, float* pre,
                                          float* post) {
  CsrRow r{0, false, pre, post};
  if (!co.off) return r;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) r.o += part[w];
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    co.off[row] = r.o;
    if (row == co.batch - 1) co.off[co.batch] = r.o + n;
  }
  r.direct = r.o + n <= co.capacity;
  if (r.direct && co.pre) r.pre = co.pre + r.o;
  if (r.direct && co.act) r.act = co.act + r.o;
  return r;
}
// The head of a row that does not fit, each thread the entries a0, a0 + astep, ...
__device__ __forceinline__ void csr_spill(const CsrOut& co, const CsrRow& r, int n, int a0, int astep) {
  if (!co.off || r.direct) return;
  for (int a = a0; a < n && r.o + a < co.capacity; a += astep) {
    if (co.pre) co.pre[r.o + a] = r.pre[a];
    if (co.act) co.act[r.o + a] = r.act[a];
  }
}

// Latency bound: few waves, each a chain of loads.  So a row of x is read kRowLoads
// values a thread at a time and its nonzeros placed by ballots and one barrier, and
// with transposed weights those of kEntries nonzeros are in flight while the ones before
// them are summed (the list is padded to 2 * kEntries entries, whose products are replaced
// by -0.0).  With row-major weights each lane walks a row of its own, and entries in flight
// keep more lines than the 32 KB cache of a CU holds: a plain loop there (softmax of
// 100000 neurons, 64 rows of 256 inputs, 30% nonzeros: 315 us, 442 with sixteen in flight, 334
// with four).
// 128 rows of 784, 1024 neurons: 14.2 us (16.5 with 64-bit offsets), 20 with a block
// scan per 256 values of x and loads where they are used.
constexpr int kRowLoads = 4;

// The nonzeros of xr[0..dim) in ascending order, d * mul to nzi and values to nzv;
// returns their count.  wcnt: LOADS words per wave.  A barrier follows before the lists are
// read.  LOADS: values a thread reads at a time, one where the block covers the row (5000 rows
// of 30 inputs, 500 neurons: 83.5 us, 92 with four).
template <int LOADS>
__device__ __forceinline__ int row_nonzeros(const float* __restrict__ xr, int dim, uint32_t mul, uint32_t* nzi,
                                            float* nzv, int* wcnt) {
  const int waves = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int base = 0;
  for (int c0 = 0; c0 < dim; c0 += LOADS * blockDim.x) {
    float v[LOADS];
    uint64_t m[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; ++u) v[u] = xr[min(c0 + u * (int)blockDim.x + (int)threadIdx.x, dim - 1)];
    if (c0) __syncthreads();   // the counts before these have been read
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      m[u] = __ballot(c0 + u * (int)blockDim.x + (int)threadIdx.x < dim && v[u] != 0.0f);
      if (lane == 0) wcnt[u * waves + wave] = __popcll(m[u]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      int pos = base;
      for (int w = 0; w < waves; ++w) {
        const int q = wcnt[u * waves + w];
        pos += w < wave ? q : 0;
        base += q;
      }
      if ((m[u] >> lane) & 1ull) {
        pos += __popcll(m[u] & ((1ull << lane) - 1ull));
        nzi[pos] = (uint32_t)(c0 + u * (int)blockDim.x + (int)threadIdx.x) * mul;
        nzv[pos] = v[u];
      }
    }
  }
  return base;
}

// Softmax over a row's active set (layer.rs:286-308) from prow to orow, by a block of at
// least kSlideThreads threads; lmax: the thread's largest value.  The sum keeps one
// order: thread t < kSlideThreads adds entries t, t + kSlideThreads, ..., then waves,
// then the block.  kSmLoads values are in flight, and the exponentials stay in LDS (eb,
// room for ecap; free once every thread is here) between the passes, where each value
// and pass was a round trip to the caches.
constexpr int kSmLoads = 8;
__device__ __forceinline__ void softmax_row(float lmax, const float* prow, float* orow, int n, float* red, float* eb,
                                            int ecap) {
  constexpr int kWaves = kSlideThreads / 64;
  const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  lmax = wave_max(lmax);
  if ((threadIdx.x & 63) == 0) red[wave] = lmax;
  __syncthreads();
  float mx = red[0];
  for (int i = 1; i < waves; ++i) mx = fmaxf(mx, red[i]);
  __syncthreads();
  float* e_out = n <= ecap ? eb : orow;
  if (wave < kWaves) {
    float ls = 0.0f;
    for (int a = threadIdx.x; a < n; a += kSlideThreads * kSmLoads) {
      float z[kSmLoads];
#pragma unroll
      for (int u = 0; u < kSmLoads; ++u) z[u] = prow[min(a + u * kSlideThreads, n - 1)];
#pragma unroll
      for (int u = 0; u < kSmLoads; ++u) {
        if (a + u * kSlideThreads < n) {
          const float e = expf_glibc(z[u] - mx);
          e_out[a + u * kSlideThreads] = e;
          ls += e;
        }
      }
    }
    ls = wave_sum(ls);
    if ((threadIdx.x & 63) == 0) red[wave] = ls;
  }
  __syncthreads();
  float tot = 0.0f;
  for (int i = 0; i < kWaves; ++i) tot += red[i];
  const float uniform = 1.0f / (float)n;
  for (int a = threadIdx.x; a < n; a += blockDim.x) orow[a] = tot > 0.0f ? e_out[a] / tot : uniform;
}

// LOADS: row_nonzeros' (dense inputs).
template <bool SPARSE, bool TRANS, int LOADS>
__global__ __launch_bounds__(kSlideThreads) void neuron_kernel(
    const float* __restrict__ W, int nn, const float* __restrict__ bias, int dim,
    const float* __restrict__ x, const int64_t* __restrict__ xoff,
    const uint32_t* __restrict__ xidx, const float* __restrict__ xval,
    uint32_t* __restrict__ aids, int astride, const int32_t* __restrict__ alen, int act,
    int max_nz, float* __restrict__ pre, float* __restrict__ post, int fb_n,
    int32_t* __restrict__ alen_out, CsrOut co) {
  extern __shared__ unsigned char smem[];   // max_nz: a multiple of 2 * kEntries
  uint32_t* nzi = reinterpret_cast<uint32_t*>(smem);
  float* nzv = reinterpret_cast<float*>(smem + sizeof(uint32_t) * max_nz);
  __shared__ int wcnt[LOADS * (kSlideThreads / 64)];
  __shared__ float red[kSlideThreads / 64];
  __shared__ long long part[kSlideThreads / 64];
  const int64_t row = blockIdx.x;
  bool all;
  const int n = vanilla_len(alen, row, fb_n, all);
  csr_part(co, alen, row, fb_n, part);
  const bool fit = TRANS && offsets_fit(dim, nn);
  const uint32_t mul = fit ? (uint32_t)nn : 1u;   // of the indices in LDS
  int nnz;
  int64_t xa = 0;
  if (SPARSE) {
    xa = xoff[row];
    nnz = (int)(xoff[row + 1] - xa);
    if (nnz <= max_nz)
      for (int i = threadIdx.x; i < nnz; i += blockDim.x) {
        nzi[i] = xidx[xa + i] * mul;
        nzv[i] = xval[xa + i];
      }
  } else {
    nnz = row_nonzeros<LOADS>(x + row * (int64_t)dim, dim, mul, nzi, nzv, wcnt);
  }
  const bool in_lds = !SPARSE || nnz <= max_nz;
  const int npad = entries_padded(nnz);
  if (in_lds)
    for (int i = nnz + threadIdx.x; i < npad; i += blockDim.x) {
      nzi[i] = 0u;
      nzv[i] = 0.0f;
    }
  __syncthreads();
  uint32_t* ids = aids + row * (int64_t)astride;
  const CsrRow cr = csr_row(co, row, n, part, pre + row * (int64_t)astride, post + row * (int64_t)astride);
  float *prow = cr.pre, *orow = cr.act;
  if (alen_out && blockIdx.y == 0 && threadIdx.x == 0) alen_out[row] = n;
  float lmax = -INFINITY;
  const int a0 = threadIdx.x + blockIdx.y * blockDim.x, astep = blockDim.x * gridDim.y;
  for (int a = a0; a < n; a += astep) {
    const uint32_t id = all ? (uint32_t)a : ids[a];
    if (!co.off) {
      if (all) ids[a] = id;
    } else if (cr.o + a < co.capacity) {
      co.ids[cr.o + a] = id;
    }
    const float bi = bias[id];
    const float* __restrict__ wl = TRANS ? W + id : W + (size_t)id * dim;   // this lane's weights
    float s = -0.0f;
    if (in_lds && !TRANS) {
      for (int e = 0; e < nnz; ++e) s = __fadd_rn(s, __fmul_rn(wl[nzi[e]], nzv[e]));
    } else if (in_lds && nnz && fit) {
      s = sum_entries(nzi, nzv, nnz, [&](uint32_t q) { return weight_at(W, id + q); });
    } else if (in_lds && nnz) {
      s = sum_entries(nzi, nzv, nnz, [&](uint32_t d) { return wl[(size_t)d * nn]; });
    } else {
      for (int e = 0; e < nnz; ++e) {
        const size_t d = xidx[xa + e];
        s = __fadd_rn(s, __fmul_rn(wl[TRANS ? d * nn : d], xval[xa + e]));
      }
    }
    const float z = __fadd_rn(s, bi);
    prow[a] = z;
    lmax = fmaxf(lmax, z);
    if (act == KH_ACT_RELU) orow[a] = fmaxf(z, 0.0f);
    else if (act == KH_ACT_SIGMOID) orow[a] = sigmoid_ref(z);
    else if (act == KH_ACT_TANH) orow[a] = tanhf(z);
    else if (act != KH_ACT_SOFTMAX) orow[a] = z;
  }
  if (act != KH_ACT_SOFTMAX) return csr_spill(co, cr, n, a0, astep);
  softmax_row(lmax, prow, orow, n, red, reinterpret_cast<float*>(smem), 2 * max_nz);
  csr_spill(co, cr, n, threadIdx.x, blockDim.x);   // its own entries (one block per row)
}

// Row-major layers over dense inputs of at most kTileMaxDim features (cfg5's
// output layer): each wave takes 32 active neurons at a time and loads their
// weight rows cooperatively, 32 lanes per 512-byte row (two whole rows per load
// instruction, instead of 64 scattered rows per instruction), into an LDS tile
// whose odd row stride makes the per-lane column reads conflict-free; lane j
// then runs neuron j's sequential sum over the input's nonzeros (ascending, as
// neuron_kernel does).  The next tile's loads are in flight during the sums, which
// have to be shorter than those loads take: sixteen LDS reads are in flight ahead of
// them.  Two waves per SIMD, so that loads also run while one of them fills its tile
// (a tile of 64, which has a lane for every lane, leaves room for one).
// 256 rows of 128, 6400 of 670091 neurons each: 135 us (6.2 TB/s); 147 us with tiles of
// 64 and a round trip per value in the softmax, 158 with each product read where it is
// added.
// With several blocks per row (gridDim.y) the tiles are dealt over them and a
// softmax layer's activations are left to another kernel; `dense`, when given,
// also gets the activations at their ids.
constexpr int kTileN = 32;
constexpr int kTileStride = 129;   // floats per LDS row
constexpr int kTileMaxDim = 128;
constexpr int kTileWaves = 8;      // waves per block at most (two at least)
constexpr int kTileThreads = 64 * kTileWaves;
constexpr size_t tile_lds(int waves) { return sizeof(float) * waves * kTileN * kTileStride; }

__global__ __launch_bounds__(kTileThreads) void neuron_tile_kernel(
    const float* __restrict__ W, const float* __restrict__ bias, int dim, const float* __restrict__ x,
    uint32_t* __restrict__ aids, int astride, const int32_t* __restrict__ alen, int act,
    float* __restrict__ pre, float* __restrict__ post, int fb_n, int32_t* __restrict__ alen_out,
    float* __restrict__ dense, int64_t dense_ld, CsrOut co) {
  extern __shared__ float tl[];
  __shared__ uint32_t nzi[kTileMaxDim];   // a multiple of 2 * kEntries
  __shared__ float nzv[kTileMaxDim];
  __shared__ int wcnt[kTileWaves];
  __shared__ float red[kTileWaves];
  __shared__ long long part[kTileWaves];
  const int64_t row = blockIdx.x;
  const int waves = blockDim.x >> 6;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  csr_part(co, alen, row, fb_n, part);
  const int nnz = row_nonzeros<1>(x + row * (int64_t)dim, dim, 1u, nzi, nzv, wcnt);   // dim <= 128 <= blockDim
  for (int i = nnz + threadIdx.x; i < entries_padded(nnz); i += blockDim.x) {
    nzi[i] = 0u;
    nzv[i] = 0.0f;
  }
  __syncthreads();
  bool all;
  const int n = vanilla_len(alen, row, fb_n, all);
  uint32_t* ids = aids + row * (int64_t)astride;
  const CsrRow cr = csr_row(co, row, n, part, pre + row * (int64_t)astride, post + row * (int64_t)astride);
  float *prow = cr.pre, *orow = cr.act;
  if (alen_out && blockIdx.y == 0 && threadIdx.x == 0) alen_out[row] = n;
  if (all && !co.off && blockIdx.y == 0)
    for (int a = threadIdx.x; a < n; a += blockDim.x) ids[a] = (uint32_t)a;
  float* buf = tl + (size_t)wave * kTileN * kTileStride;
  const int q4 = dim >> 2;              // float4 per weight row (<= 32)
  const int c = lane & 31;              // this lane's float4 of a row, and its neuron of a tile
  const int half = lane >> 5;           // which of the two rows of a load
  const int ntiles = (n + kTileN - 1) / kTileN;
  float4 v[kTileN / 2];
  // neuron c of tile t (clamped to the last active id), the same in both halves
  auto id_of = [&](int t) {
    const int ia = min(t * kTileN + c, n - 1);
    return all ? (uint32_t)ia : ids[ia];
  };
  // the rows of the next tile, whose ids came with the one before it
  uint32_t id_next = 0u, id_tile = 0u;
  float b_tile = 0.0f;
  auto issue = [&](int t_next) {
    id_tile = id_next;
    b_tile = bias[id_tile];
    id_next = id_of(t_next);
#pragma unroll
    for (int r = 0; r < kTileN / 2; ++r) {
      const uint32_t id = (uint32_t)__shfl((int)id_tile, 2 * r + half);
      v[r] = reinterpret_cast<const float4*>(W + (size_t)id * dim)[min(c, q4 - 1)];
    }
  };
  float lmax = -INFINITY;
  int t = (int)blockIdx.y * waves + wave;
  const int tstep = (int)gridDim.y * waves;
  if (t < ntiles) {
    id_next = id_of(t);
    issue(t + tstep);
  }
  for (; t < ntiles; t += tstep) {
    const uint32_t id = id_tile;
    const float bi = b_tile;
    // the tile to LDS (column 4c..4c+3 of row 2r + half)
    if (c < q4) {
#pragma unroll
      for (int r = 0; r < kTileN / 2; ++r) {
        float* dst = buf + (2 * r + half) * kTileStride + 4 * c;
        dst[0] = v[r].x;
        dst[1] = v[r].y;
        dst[2] = v[r].z;
        dst[3] = v[r].w;
      }
    }
    if (t + tstep < ntiles) issue(t + 2 * tstep);
    const int a = t * kTileN + c;
    const float* wr = buf + c * kTileStride;
    const float s = nnz ? sum_entries(nzi, nzv, nnz, [&](uint32_t d) { return wr[d]; }) : -0.0f;
    if (a < n && half == 0) {
      const float z = __fadd_rn(s, bi);
      prow[a] = z;
      if (co.off && cr.o + a < co.capacity) co.ids[cr.o + a] = id;
      lmax = fmaxf(lmax, z);
      if (act != KH_ACT_SOFTMAX) {
        float r;
        if (act == KH_ACT_RELU) r = fmaxf(z, 0.0f);
        else if (act == KH_ACT_SIGMOID) r = sigmoid_ref(z);
        else if (act == KH_ACT_TANH) r = tanhf(z);
        else r = z;
        orow[a] = r;
        if (dense) dense[row * dense_ld + id] = r;
      }
    }
  }
  if (act != KH_ACT_SOFTMAX || gridDim.y > 1) {
    if (!co.off || cr.direct) return;
    __syncthreads();   // the entries are other lanes'
    return csr_spill(co, cr, n, threadIdx.x, blockDim.x);   // (one block per row with a CsrOut)
  }
  softmax_row(lmax, prow, orow, n, red, tl, waves * kTileN * kTileStride);
  csr_spill(co, cr, n, threadIdx.x, blockDim.x);
}

// neuron_tile_kernel's LDS (above 64 KB) is allowed once per process.
static int tile_kernel_ready() {
  static std::once_flag once;
  static int rc = KH_OK;
  std::call_once(once, [] {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&neuron_tile_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_lds(kTileWaves)) != hipSuccess)
      rc = KH_ERR_HIP;
  });
  return rc;
}

bool neuron_tile_ok(const kh_slide_layer* l) {
  return l->dim <= kTileMaxDim && l->dim % 4 == 0 && tile_kernel_ready() == KH_OK;
}

// Two waves a block (a tile each): the few tiles of a short batch spread over as
// many CUs as there are.  At least two blocks a row, so a softmax stays undone.
int neuron_tile_launch(const kh_slide_layer* l, const float* x, int64_t rows, uint32_t* aids, int as,
                       const int32_t* alen, float* pre, float* post, float* dense, int64_t dense_ld,
                       hipStream_t st) {
  constexpr int kFew = 2;
  const int tiles = ceil_div(as, kTileN * kFew);
  const int split = std::max(2, std::min(tiles, std::max(1, 1024 / (int)std::min<int64_t>(rows, 1024))));
  hipLaunchKernelGGL(neuron_tile_kernel, dim3((unsigned)rows, (unsigned)split), dim3(64 * kFew), tile_lds(kFew), st,
                     l->w, l->bias, l->dim, x, aids, as, alen, l->act, pre, post, 0, nullptr, dense,
                     dense_ld, CsrOut{});
  KH_LAUNCHED();
  return KH_OK;
}

// Dense layer over CSR inputs: y[b][o] = act(sum_e val_e * W^T[idx_e][o] + bias[o]).
constexpr int kChainBatch = 16;  // entries in flight per sequential sum
__global__ __launch_bounds__(256) void dense_sparse_kernel(const float* __restrict__ WT, int n,
                                                           const float* __restrict__ bias,
                                                           const int64_t* __restrict__ xoff,
                                                           const uint32_t* __restrict__ xidx,
                                                           const float* __restrict__ xval,
                                                           int act, float* __restrict__ y) {
  const int64_t row = blockIdx.y;
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= n) return;
  const int64_t a = xoff[row], b = xoff[row + 1];
  // kChainBatch entries at a time (indices, then the weight rows, all in
  // flight), then added in order: the sum stays sequential
  float s = -0.0f;
  for (int64_t e0 = a; e0 < b; e0 += kChainBatch) {
    uint32_t ix[kChainBatch];
    float xv[kChainBatch], wv[kChainBatch];
#pragma unroll
    for (int j = 0; j < kChainBatch; ++j) {
      const int64_t e = min(e0 + j, b - 1);
      ix[j] = xidx[e];
      xv[j] = xval[e];
    }
#pragma unroll
    for (int j = 0; j < kChainBatch; ++j) wv[j] = WT[(size_t)ix[j] * n + o];
#pragma unroll
    for (int j = 0; j < kChainBatch; ++j)
      if (e0 + j < b) s = __fadd_rn(s, __fmul_rn(xv[j], wv[j]));
  }
  const float z = __fadd_rn(s, bias[o]);
  float r;
  if (act == KH_ACT_RELU) r = fmaxf(z, 0.0f);
  else if (act == KH_ACT_SIGMOID) r = sigmoid_ref(z);
  else if (act == KH_ACT_TANH) r = tanhf(z);
  else r = z;
  y[row * (int64_t)n + o] = r;
}

int select_launch_with(const kh_lsh_index* idx, int sampling, int top_k, int threshold,
                       int num_neurons, const uint32_t* qids, const uint32_t* qcnt,
                       const int32_t* qlen, int qs, int64_t batch, uint32_t* aids, int as,
                       int32_t* alen, bool count_order, float* clear_dense, bool fallback,
                       hipStream_t st) {
  // A candidate's hit count is at most L * cap (every slot of its L buckets).
  const int nbins = idx->L * idx->cap + 1;
  KH_CHECK_ARG(sampling != KH_SAMPLING_TOPK || nbins <= kMaxCountBins,
               "top-k sampling supports num_tables * bucket_capacity <= %d", kMaxCountBins - 1);
  hipLaunchKernelGGL(select_kernel, dim3((unsigned)batch),
                     dim3(batch <= kSelectFewRows ? kSelectThreads : kSlideThreads),
                     sampling == KH_SAMPLING_TOPK ? sizeof(unsigned) * nbins : 0, st, qids, qcnt,
                     qlen, qs, sampling, top_k, threshold, num_neurons, nbins, aids, as, alen,
                     count_order ? 1 : 0, clear_dense, fallback ? 1 : 0,
                     idx->id_bound <= (uint32_t)num_neurons ? 1 : 0);
  KH_LAUNCHED();
  return KH_OK;
}

int select_launch(const kh_slide_layer* l, const uint32_t* qids, const uint32_t* qcnt,
                  const int32_t* qlen, int qs, int64_t batch, uint32_t* aids, int as, int32_t* alen,
                  bool count_order, float* clear_dense, hipStream_t st) {
  return select_launch_with(l->index, l->sampling, l->top_k, l->threshold, l->n, qids, qcnt, qlen,
                            qs, batch, aids, as, alen, count_order, clear_dense, true, st);
}

}  // namespace kh

using namespace kh;

struct kh_dense_layer {
  int dim = 0, n = 0, act = 0;
  float* wt = nullptr;  // [dim][n]
  float* bias = nullptr;
};

extern "C" int kh_slide_layer_create(int input_dim, int num_neurons, const float* w_host,
                                     const float* bias_host, kh_lsh_index* index, int sampling,
                                     int top_k, int threshold, int activation,
                                     kh_slide_layer** out) {
  KH_CHECK_ARG(out && w_host && bias_host && index, "null argument");
  KH_CHECK_ARG(input_dim > 0 && num_neurons > 0, "dims must be positive");
  KH_CHECK_ARG(index->h->dim == input_dim, "index input_dim %d != layer input_dim %d",
               index->h->dim, input_dim);
  KH_CHECK_ARG(sampling >= 0 && sampling <= 2 && activation >= 0 && activation <= 4,
               "bad sampling / activation");
  KH_CHECK_ARG(top_k >= 0 && threshold >= 0, "bad top_k / threshold");
  *out = nullptr;
  auto* l = new kh_slide_layer();
  l->dim = input_dim;
  l->n = num_neurons;
  l->index = index;
  l->sampling = sampling;
  l->top_k = top_k;
  l->threshold = threshold;
  l->act = activation;
  const size_t nw = (size_t)input_dim * num_neurons;
  l->w = static_cast<float*>(dev_alloc(sizeof(float) * nw));
  l->bias = static_cast<float*>(dev_alloc(sizeof(float) * num_neurons));
  uint32_t* ids = static_cast<uint32_t*>(dev_alloc(sizeof(uint32_t) * num_neurons));
  int rc = (l->w && l->bias && ids) ? KH_OK : KH_ERR_ALLOC;
  if (rc == KH_OK) {
    std::vector<uint32_t> h(num_neurons);
    for (int i = 0; i < num_neurons; ++i) h[i] = (uint32_t)i;
    if (hipMemcpy(l->w, w_host, sizeof(float) * nw, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(l->bias, bias_host, sizeof(float) * num_neurons, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(ids, h.data(), sizeof(uint32_t) * num_neurons, hipMemcpyHostToDevice) != hipSuccess) {
      set_error("layer upload failed");
      rc = KH_ERR_HIP;
    }
  }
  // Transposed copy [dim][n] for the neuron kernel of non-softmax layers: the
  // lanes of a wave take ascending active ids, so one load instruction reads a
  // few adjacent cache lines of one input row instead of 64 weight rows.
  if (rc == KH_OK && activation != KH_ACT_SOFTMAX) {
    l->wtn = static_cast<float*>(dev_alloc(sizeof(float) * nw));
    if (!l->wtn) rc = KH_ERR_ALLOC;
    if (rc == KH_OK) {
      hipLaunchKernelGGL(transpose_kernel<float>, dim3(ceil_div(input_dim, 32), ceil_div(num_neurons, 32)),
                         dim3(256), 0, 0, l->w, num_neurons, input_dim, l->wtn);
      if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
        set_error("layer transpose failed");
        rc = KH_ERR_HIP;
      }
    }
  }
  // Layer::new inserts neurons 0..n-1 in order (layer.rs:42-44).
  if (rc == KH_OK) rc = kh_lsh_index_insert(index, ids, l->w, num_neurons, input_dim, nullptr);
  dev_free(ids);
  if (rc != KH_OK) {
    kh_slide_layer_destroy(l);
    return rc;
  }
  *out = l;
  return KH_OK;
}

extern "C" int kh_slide_layer_destroy(kh_slide_layer* l) {
  if (!l) return KH_OK;
  dev_free(l->w);
  dev_free(l->wtn);
  dev_free(l->bias);
  l->free_opt();
  delete l;
  return KH_OK;
}

// Sampling as a SparseInferenceEngine call makes it (bolt/sparse_inference.rs):
// top-k by count in the sampler's order, no all-neurons fallback, and its own
// activation.
struct SelectOverride {
  int top_k;
  int act;
};

static int slide_forward_common(const kh_slide_layer* lc, const float* x, const int64_t* xoff,
                                const uint32_t* xidx, const float* xval, int64_t batch,
                                int64_t* off, uint32_t* act_ids, float* pre_out, float* act_out,
                                int64_t capacity, hipStream_t st,
                                const SelectOverride* ov = nullptr) {
  const kh_slide_layer* l = lc;
  const kh_lsh_index* idx = l->index;
  const int L = idx->L;
  WsSet* w = l->ws.get(st);
  uint32_t* codes = static_cast<uint32_t*>(w->get(0, sizeof(uint32_t) * batch * L));
  // Vanilla sampling with every indexed id below the layer's neuron count
  // keeps the whole query result (layer.rs:65-90), so the neuron kernel reads
  // it directly and applies the empty-set fallback itself: no select launch.
  const bool direct = !ov && l->sampling == KH_SAMPLING_VANILLA && idx->id_bound <= (uint32_t)l->n;
  const int qs = direct ? std::max(query_stride(idx), l->n) : query_stride(idx);
  uint32_t* qids = static_cast<uint32_t*>(w->get(1, sizeof(uint32_t) * batch * qs));
  uint32_t* qcnt = static_cast<uint32_t*>(w->get(2, sizeof(uint32_t) * batch * qs));
  int32_t* qlen = static_cast<int32_t*>(w->get(3, sizeof(int32_t) * batch));
  const int as = std::max(qs, l->n);
  uint32_t* aids = static_cast<uint32_t*>(w->get(4, sizeof(uint32_t) * batch * as));
  int32_t* alen = static_cast<int32_t*>(w->get(5, sizeof(int32_t) * batch));
  const bool packed = batch <= kCsrPackMax;   // the kernel writes the CSR rows itself
  const bool spill = !(packed && pre_out && act_out && capacity >= batch * (int64_t)as);
  float* pre = spill ? static_cast<float*>(w->get(6, sizeof(float) * batch * as)) : nullptr;
  float* post = spill ? static_cast<float*>(w->get(7, sizeof(float) * batch * as)) : nullptr;
  if (!codes || !qids || !qcnt || !qlen || !aids || !alen || (spill && (!pre || !post))) return KH_ERR_ALLOC;
  int rc = xoff ? hash_sparse_launch(idx->h, xoff, xidx, xval, batch, codes, st)
                : hash_dense_launch(idx->h, x, l->dim, batch, codes, st);
  if (rc != KH_OK) return rc;
  rc = query_launch(idx, codes, batch, qids, direct ? nullptr : qcnt, qs, qlen, st);
  if (rc != KH_OK) return rc;
  if (direct)
    aids = qids;  // stride qs == as
  else
    rc = ov ? select_launch_with(l->index, KH_SAMPLING_TOPK, ov->top_k, 0, l->n, qids, qcnt, qlen, qs,
                                 batch, aids, as, alen, true, nullptr, false, st)
            : select_launch(l, qids, qcnt, qlen, qs, batch, aids, as, alen, false, nullptr, st);
  if (rc != KH_OK) return rc;
  const int act = ov ? ov->act : l->act;
  const int max_nz = xoff ? 4096 : entries_padded(l->dim);
  KH_CHECK_ARG(xoff || l->dim <= 8192, "dense SLIDE input supports input_dim <= 8192");
  const size_t lds = (sizeof(uint32_t) + sizeof(float)) * max_nz;
  // Without softmax the active ids of a sample are split over up to kNeuronSplit
  // blocks (softmax needs the whole row's max and sum in one block); a block lists
  // the row's nonzeros first, so there are none without ids (5000 rows of 20
  // neurons: 57 us, 86 with four blocks each).
  constexpr int kNeuronSplit = 4;
  const dim3 ng((unsigned)batch, l->wtn ? (unsigned)std::min(kNeuronSplit, ceil_div(as, kSlideThreads)) : 1u);
  // direct: the candidate lengths come from the query, the fallback is the
  // kernel's, and the kernel writes the lengths the outputs use
  const int32_t* ilen = direct ? qlen : alen;
  const int fb_n = direct ? l->n : 0;
  int32_t* olen = direct && !packed ? alen : nullptr;
  const bool wide = l->dim > kSlideThreads;
  CsrOut co{};
  if (packed) co = {off, act_ids, pre_out, act_out, batch, capacity};
  if (xoff && l->wtn)
    hipLaunchKernelGGL((neuron_kernel<true, true, 1>), ng, dim3(kSlideThreads), lds, st, l->wtn, l->n,
                       l->bias, l->dim, nullptr, xoff, xidx, xval, aids, as, ilen, act, max_nz,
                       pre, post, fb_n, olen, co);
  else if (xoff)
    hipLaunchKernelGGL((neuron_kernel<true, false, 1>), ng, dim3(kSlideThreads), lds, st, l->w, l->n,
                       l->bias, l->dim, nullptr, xoff, xidx, xval, aids, as, ilen, act, max_nz,
                       pre, post, fb_n, olen, co);
  else if (l->wtn)
    hipLaunchKernelGGL((wide ? neuron_kernel<false, true, kRowLoads> : neuron_kernel<false, true, 1>), ng,
                       dim3(kSlideThreads), lds, st, l->wtn, l->n, l->bias, l->dim, x, nullptr, nullptr, nullptr, aids,
                       as, ilen, act, max_nz, pre, post, fb_n, olen, co);
  else if (l->dim <= kTileMaxDim && l->dim % 4 == 0 && tile_kernel_ready() == KH_OK) {
    // Eight waves are a block per CU. Rows without a tile for each take the four that the
    // softmax needs, two blocks to a CU: 5000 rows of 20 neurons 94 us, 163 with eight.
    const int waves = ceil_div(as, kTileN) < kTileWaves ? kSlideThreads / 64 : kTileWaves;
    hipLaunchKernelGGL(neuron_tile_kernel, dim3((unsigned)batch), dim3(64 * waves), tile_lds(waves), st, l->w, l->bias,
                       l->dim, x, aids, as, ilen, act, pre, post, fb_n, olen, nullptr, 0, co);
  }
  else
    hipLaunchKernelGGL((wide ? neuron_kernel<false, false, kRowLoads> : neuron_kernel<false, false, 1>), ng,
                       dim3(kSlideThreads), lds, st, l->w, l->n, l->bias, l->dim, x, nullptr, nullptr, nullptr, aids,
                       as, ilen, act, max_nz, pre, post, fb_n, olen, co);
  KH_LAUNCHED();
  if (packed) return csr_check(off, batch, as, capacity, st);
  return csr_finish(aids, nullptr, pre, post, as, alen, batch, off, act_ids, nullptr, pre_out,
                    act_out, capacity, st);
}

extern "C" int kh_slide_layer_forward(const kh_slide_layer* l, const float* x_dev, int64_t batch,
                                      int64_t* off_dev, uint32_t* act_ids_dev, float* pre_dev,
                                      float* act_dev, int64_t capacity, void* stream) {
  KH_CHECK_ARG(l && off_dev && act_ids_dev, "null argument");
  KH_CHECK_ARG(batch >= 0 && batch <= 0x7fffffff && capacity >= 0, "bad batch/capacity");
  hipStream_t st = as_stream(stream);
  if (batch == 0) {
    KH_HIP(hipMemsetAsync(off_dev, 0, sizeof(int64_t), st));
    return KH_OK;
  }
  KH_CHECK_ARG(x_dev != nullptr, "null input");
  return slide_forward_common(l, x_dev, nullptr, nullptr, nullptr, batch, off_dev, act_ids_dev,
                              pre_dev, act_dev, capacity, st);
}

extern "C" int kh_slide_layer_forward_sparse(const kh_slide_layer* l, const int64_t* xoff_dev,
                                             const uint32_t* xidx_dev, const float* xval_dev,
                                             int64_t batch, int64_t* off_dev,
                                             uint32_t* act_ids_dev, float* pre_dev, float* act_dev,
                                             int64_t capacity, void* stream) {
  KH_CHECK_ARG(l && off_dev && act_ids_dev && xoff_dev, "null argument");
  KH_CHECK_ARG(batch >= 0 && batch <= 0x7fffffff && capacity >= 0, "bad batch/capacity");
  hipStream_t st = as_stream(stream);
  if (batch == 0) {
    KH_HIP(hipMemsetAsync(off_dev, 0, sizeof(int64_t), st));
    return KH_OK;
  }
  return slide_forward_common(l, nullptr, xoff_dev, xidx_dev, xval_dev, batch, off_dev,
                              act_ids_dev, pre_dev, act_dev, capacity, st);
}

extern "C" int kh_sparse_inference(const kh_slide_layer* l, const float* x_dev, int64_t batch,
                                   int64_t base_top_k, float sparsity_multiplier, int relu,
                                   int64_t* off_dev, uint32_t* ids_dev, float* act_dev,
                                   int64_t capacity, void* stream) {
  KH_CHECK_ARG(l && off_dev && ids_dev, "null argument");
  KH_CHECK_ARG(batch >= 0 && batch <= 0x7fffffff && capacity >= 0 && base_top_k >= 0,
               "bad batch/capacity/top_k");
  hipStream_t st = as_stream(stream);
  if (batch == 0) {
    KH_HIP(hipMemsetAsync(off_dev, 0, sizeof(int64_t), st));
    return KH_OK;
  }
  KH_CHECK_ARG(x_dev != nullptr, "null input");
  // (base_top_k as f32 * multiplier) as usize: f32 product, truncated,
  // saturating (NaN and negatives give 0)
  const float ek = static_cast<float>(base_top_k) * sparsity_multiplier;
  const int64_t eff = !(ek > 0.0f) ? 0 : (ek >= 2147483647.0f ? 0x7fffffff : static_cast<int64_t>(ek));
  SelectOverride ov{static_cast<int>(eff), relu ? KH_ACT_RELU : KH_ACT_IDENTITY};
  return slide_forward_common(l, x_dev, nullptr, nullptr, nullptr, batch, off_dev, ids_dev, nullptr,
                              act_dev, capacity, st, &ov);
}

extern "C" int kh_lsh_index_query_top_k(const kh_lsh_index* idx, const float* x_dev, int64_t batch,
                                        int64_t top_k, uint32_t* ids_dev, int32_t* n_dev,
                                        void* stream) {
  KH_CHECK_ARG(idx && n_dev && (ids_dev || top_k == 0), "null argument");
  KH_CHECK_ARG(batch >= 0 && batch <= 0x7fffffff && top_k >= 0 && top_k <= 0x7fffffff, "bad batch/top_k");
  if (batch == 0) return KH_OK;
  KH_CHECK_ARG(x_dev != nullptr, "null input");
  hipStream_t st = as_stream(stream);
  WsSet* w = idx->ws.get(st);
  const int L = idx->L;
  const int qs = query_stride(idx);
  uint32_t* codes = static_cast<uint32_t*>(w->get(4, sizeof(uint32_t) * batch * L));
  uint32_t* qids = static_cast<uint32_t*>(w->get(5, sizeof(uint32_t) * batch * qs));
  uint32_t* qcnt = static_cast<uint32_t*>(w->get(6, sizeof(uint32_t) * batch * qs));
  int32_t* qlen = static_cast<int32_t*>(w->get(7, sizeof(int32_t) * batch));
  if (!codes || !qids || !qcnt || !qlen) return KH_ERR_ALLOC;
  int rc = hash_dense_launch(idx->h, x_dev, idx->h->dim, batch, codes, st);
  if (rc == KH_OK) rc = query_launch(idx, codes, batch, qids, qcnt, qs, qlen, st);
  if (rc != KH_OK) return rc;
  // count descending, then id, straight into the caller's [batch][top_k]
  // rows: the count-order selection writes only positions below
  // min(top_k, candidates)
  const int k = static_cast<int>(std::min<int64_t>(top_k, qs));
  return select_launch_with(idx, KH_SAMPLING_TOPK, k, 0, 0x7fffffff, qids, qcnt, qlen, qs, batch, ids_dev,
                            static_cast<int>(top_k), n_dev, true, nullptr, false, st);
}

extern "C" int kh_dense_layer_create(int input_dim, int num_neurons, const float* w_host,
                                     const float* bias_host, int activation,
                                     kh_dense_layer** out) {
  KH_CHECK_ARG(out && w_host && bias_host, "null argument");
  KH_CHECK_ARG(input_dim > 0 && num_neurons > 0 && activation >= 0 && activation <= 4 &&
                   activation != KH_ACT_SOFTMAX,
               "bad dims / activation (softmax is not supported on a dense layer)");
  *out = nullptr;
  auto* l = new kh_dense_layer();
  l->dim = input_dim;
  l->n = num_neurons;
  l->act = activation;
  const size_t nw = (size_t)input_dim * num_neurons;
  std::vector<float> wt(nw);
  for (int o = 0; o < num_neurons; ++o)
    for (int d = 0; d < input_dim; ++d) wt[(size_t)d * num_neurons + o] = w_host[(size_t)o * input_dim + d];
  l->wt = static_cast<float*>(dev_alloc(sizeof(float) * nw));
  l->bias = static_cast<float*>(dev_alloc(sizeof(float) * num_neurons));
  if (!l->wt || !l->bias) {
    kh_dense_layer_destroy(l);
    return KH_ERR_ALLOC;
  }
  if (hipMemcpy(l->wt, wt.data(), sizeof(float) * nw, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(l->bias, bias_host, sizeof(float) * num_neurons, hipMemcpyHostToDevice) != hipSuccess) {
    set_error("dense layer upload failed");
    kh_dense_layer_destroy(l);
    return KH_ERR_HIP;
  }
  *out = l;
  return KH_OK;
}

extern "C" int kh_dense_layer_destroy(kh_dense_layer* l) {
  if (!l) return KH_OK;
  dev_free(l->wt);
  dev_free(l->bias);
  delete l;
  return KH_OK;
}

extern "C" int kh_dense_layer_forward_sparse(const kh_dense_layer* l, const int64_t* xoff_dev,
                                             const uint32_t* xidx_dev, const float* xval_dev,
                                             int64_t batch, float* y_dev, void* stream) {
  KH_CHECK_ARG(l && xoff_dev && y_dev, "null argument");
  KH_CHECK_ARG(batch >= 0 && batch <= 65535, "bad batch");
  if (batch == 0) return KH_OK;
  hipLaunchKernelGGL(dense_sparse_kernel, dim3(ceil_div(l->n, 256), (unsigned)batch), dim3(256), 0,
                     as_stream(stream), l->wt, l->n, l->bias, xoff_dev, xidx_dev, xval_dev, l->act,
                     y_dev);
  KH_LAUNCHED();
  return KH_OK;
}
