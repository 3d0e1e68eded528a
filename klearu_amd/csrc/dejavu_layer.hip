// dejavu_layer.hip -- the klearu-dejavu transformer layer's sparse MLP and
// sparse attention (f32 weights with bias) on the GPU (gfx950).
//
// Replaces Linear::forward / forward_sparse
// (crates/klearu-dejavu/src/transformer/mod.rs:114-134), SparseMlp::forward
// (crates/klearu-dejavu/src/mlp.rs:23-58) and SparseAttention::forward
// (crates/klearu-dejavu/src/attention.rs:18-74).
//
// Every output is bit-identical to the reference: each one is a sequential f32
// sum of rounded products in the reference's order, added by one lane.
//   Linear rows     per (token, output row): -0.0 + w[r][0]*x[0] + ... then
//                   + bias[r].
//   SparseMlp       gate and up rows of a selected neuron, h = silu(g) * u; then
//                   per (token, output j) W_down[j][sel[a]] * h[a] added for every
//                   selected a with h != 0, in selection order from +0.0, then the
//                   bias.
//   SparseAttention q/k/v rows of the selected heads into [heads*head_dim]
//                   vectors, a wave per (token, head) for the sigmoid score and
//                   the scaled v (zero for other heads), then o_proj over the
//                   whole (zero-filled) vector like Linear::forward.
// A handle keeps its weights twice: row-major [out][in], which the selected rows
// of a gather read in whole pieces, and transposed [in][out], which the columns
// of SparseMlp's down projection and the wide form below read.
// Index lists arrive from the host (the reference's &[usize]), are checked
// there (an out-of-range index is the reference's panic) and go to the handle's
// scratch: short ones inside a launch, longer ones by a copy that is waited for;
// either way the caller's list may be freed on return.
#include <algorithm>

#include "chain_add.hpp"
#include "gather.hpp"

struct kh_dejavu_linear {
  int in_f = 0, out_f = 0;
  float* w = nullptr;     // [out_f][in_f]
  float* wt = nullptr;    // [in_f][out_f]
  float* bias = nullptr;  // [out_f]
  mutable kh::StreamWs ws;  // forward_sparse row list, per stream
};

struct kh_dejavu_sparse_mlp {
  int hidden = 0, inter = 0;
  mutable kh::StreamWs ws;  // selected neurons and their activations, per stream
};

struct kh_dejavu_sparse_attention {
  int hidden = 0, num_heads = 0, head_dim = 0;
  mutable kh::StreamWs ws;  // row lists and head vectors, per stream
};

namespace kh {

constexpr int kDlThreads = 256;

// Few outputs: a chain of in_f dependent adds per output bounds the call (about
// 6 cycles a step), so a block gives all else to other waves.  It owns 16 rows
// x TB tokens, one chain per lane of wave 0 (the consumer); waves 1..8 hold the
// weights of the next kChainAhead chunks of kDcStep steps in registers and form a
// chunk's products in LDS while wave 0 adds the chunk before, four per read.
// Products past the end are -0.0, which leaves every sum unchanged.  A thread per
// output with one load in flight per add took 107 us for a 1024-square Linear of
// 1 to 128 tokens and 212 us at 2048 (both launch-bound here up to 16 tokens, about
// 11 us a call); SparseMlp 1024 / 2752, 30% of the neurons, 16 tokens: 668 -> 37 us,
// 1024 tokens: 11.8 -> 1.1 ms.
constexpr int kDcRows = 16;                    // output rows (or columns) per block
constexpr int kDcStep = 128;                   // steps per chunk
constexpr int kDcProd = kDcStep / 4 * kDcRows; // producer threads: one float4 of one row each
constexpr int kDcThreads = 64 + kDcProd;
// Chunks of 16 * TB chains, padded by one float4 so that the down kernel's 4-byte
// writes fall in distinct banks.
template <int TB>
using DcLds = ChainLds<kDcStep, kDcRows * TB>;

struct DcMat {
  const float* w;     // rows kernel: [out][in]; down kernel: transposed [in][out]
  const float* bias;
  float* y;
};
struct DcRows {
  DcMat m[3];         // blockIdx.z picks one; gate/up: m[0] gate, m[1] up
  int in_f;
  const float* x;     // [batch][ldx]
  int64_t ldx, batch;
  const int64_t* rows;  // null: every row
  int64_t nrows, ldy;
  int head_dim;       // 0: rows lists rows; else it lists heads of head_dim rows each
  int scatter;        // outputs at y[row] instead of y[position in the list]
};

// Output row of position `at` of the call's list.
__device__ __forceinline__ int64_t dc_row(const DcRows& a, int64_t at) {
  if (!a.rows) return at;
  if (a.head_dim == 0) return a.rows[at];
  const int64_t h = at / a.head_dim;
  return a.rows[h] * a.head_dim + (at - h * a.head_dim);
}

// Four consecutive floats at p[k..k+3], k + i < n (others read p[n - 1]).
template <bool VEC>
__device__ __forceinline__ float4 dc_load4(const float* __restrict__ p, int k, int n) {
  if constexpr (VEC) return *reinterpret_cast<const float4*>(p + min(k, n - 4));
  return make_float4(p[min(k, n - 1)], p[min(k + 1, n - 1)], p[min(k + 2, n - 1)], p[min(k + 3, n - 1)]);
}

// GATEUP: rows 0..7 of the block are gate rows, 8..15 the same neurons' up rows.
// VEC: in_f and ldx multiples of 4, x 16-byte aligned.
template <bool GATEUP, int TB, bool VEC>
__global__ __launch_bounds__(kDcThreads) void dl_chain_rows_kernel(const DcRows a) {
  __shared__ DcLds<TB> lds;
  constexpr int kOwn = GATEUP ? kDcRows / 2 : kDcRows;   // list entries per block
  const int64_t a0 = (int64_t)blockIdx.x * kOwn, b0 = (int64_t)blockIdx.y * TB;
  const int n = a.in_f, nch = (n + kDcStep - 1) / kDcStep;
  const bool prod = threadIdx.x >= 64;
  const int pt = (int)threadIdx.x - 64;
  // lanes of a producer wave: 16 rows x 4 quads, so a quad row's 16 products are
  // written as one contiguous piece per token
  const int i = prod ? pt & (kDcRows - 1) : (int)threadIdx.x & (kDcRows - 1);
  const int k4 = pt >> 4;
  const DcMat& mat = a.m[GATEUP ? i / kOwn : (int)blockIdx.z];
  const int64_t at = min(a0 + (GATEUP ? i % kOwn : i), a.nrows - 1);
  const int64_t r = dc_row(a, at);
  const float* __restrict__ wr = mat.w + r * n;
  const float* __restrict__ xr[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) xr[t] = a.x + min(b0 + t, a.batch - 1) * a.ldx;
  float4 w[kChainAhead], x[kChainAhead][TB];
  auto fetch = [&](int c, int u) {
    const int k = c * kDcStep + 4 * k4;
    w[u] = dc_load4<VEC>(wr, k, n);
#pragma unroll
    for (int t = 0; t < TB; ++t) x[u][t] = dc_load4<VEC>(xr[t], k, n);
  };
  if (prod) {
#pragma unroll
    for (int u = 0; u < kChainAhead; ++u) fetch(u, u);
  }
  float s = chain_run(lds, nch, -0.0f, [&](int c, int u) {
    const int k = c * kDcStep + 4 * k4;
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      float4 p;
      p.x = k < n ? w[u].x * x[u][t].x : -0.0f;
      p.y = k + 1 < n ? w[u].y * x[u][t].y : -0.0f;
      p.z = k + 2 < n ? w[u].z * x[u][t].z : -0.0f;
      p.w = k + 3 < n ? w[u].w * x[u][t].w : -0.0f;
      lds.q[c & 1][k4 * DcLds<TB>::kStride + t * kDcRows + i] = p;
    }
    fetch(c + kChainAhead, u);
  });
  if (threadIdx.x >= 64) return;
  const int64_t b = b0 + ((int)threadIdx.x >> 4);
  const bool live = (int)threadIdx.x < kDcRows * TB && b < a.batch;
  s = __fadd_rn(s, mat.bias[r]);
  if constexpr (GATEUP) {
    const float up = __shfl(s, (int)threadIdx.x + kOwn);
    if (live && i < kOwn && a0 + i < a.nrows) a.m[0].y[b * a.ldy + at] = __fmul_rn(silu_ref(s), up);
  } else {
    if (live && a0 + i < a.nrows) mat.y[b * a.ldy + (a.scatter ? r : at)] = s;
  }
}

// SparseMlp's down projection: chains over the selected neurons; a block owns 16
// output columns.  A producer thread takes one neuron's float4 of columns.
// VEC: hidden a multiple of 4.
template <int TB, bool VEC>
__global__ __launch_bounds__(kDcThreads) void dl_chain_down_kernel(
    const float* __restrict__ wdt, const float* __restrict__ bd, int hidden,
    const float* __restrict__ h, int64_t batch, const int64_t* __restrict__ sel, int n,
    float* __restrict__ y) {
  __shared__ DcLds<TB> lds;
  const int j0 = blockIdx.x * kDcRows;
  const int64_t b0 = (int64_t)blockIdx.y * TB;
  const int nch = (n + kDcStep - 1) / kDcStep;
  const bool prod = threadIdx.x >= 64;
  const int pt = (int)threadIdx.x - 64;
  const int q = pt & 3, e = pt >> 2;          // column quad, step within the chunk
  const float* __restrict__ hr[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) hr[t] = h + min(b0 + t, batch - 1) * n;
  int id[kChainAhead];                           // neuron of the chunk kChainAhead past the slot's
  float4 w[kChainAhead];
  float v[kChainAhead][TB];
  auto ids = [&](int c, int u) { id[u] = (int)sel[min(c * kDcStep + e, n - 1)]; };
  auto fetch = [&](int c, int u) {
    w[u] = dc_load4<VEC>(wdt + (size_t)id[u] * hidden, j0 + 4 * q, hidden);
#pragma unroll
    for (int t = 0; t < TB; ++t) v[u][t] = hr[t][min(c * kDcStep + e, n - 1)];
  };
  if (prod && nch > 0) {
#pragma unroll
    for (int u = 0; u < kChainAhead; ++u) ids(u, u);
#pragma unroll
    for (int u = 0; u < kChainAhead; ++u) fetch(u, u);
#pragma unroll
    for (int u = 0; u < kChainAhead; ++u) ids(u + kChainAhead, u);
  }
  float s = chain_run(lds, nch, 0.0f, [&](int c, int u) {
    float* dst = reinterpret_cast<float*>(&lds.q[c & 1][(e >> 2) * DcLds<TB>::kStride]) + (e & 3);
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      // a zero activation adds nothing, whatever the weight
      const bool on = c * kDcStep + e < n && v[u][t] != 0.0f;
      float* d = dst + 4 * (t * kDcRows + 4 * q);
      d[0] = on ? w[u].x * v[u][t] : -0.0f;
      d[4] = on ? w[u].y * v[u][t] : -0.0f;
      d[8] = on ? w[u].z * v[u][t] : -0.0f;
      d[12] = on ? w[u].w * v[u][t] : -0.0f;
    }
    fetch(c + kChainAhead, u);
    ids(c + 2 * kChainAhead, u);
  });
  const int lane = threadIdx.x;
  if (lane >= kDcRows * TB) return;
  const int j = j0 + (lane & (kDcRows - 1));
  const int64_t b = b0 + (lane >> 4);
  if (b < batch && j < hidden) y[b * hidden + j] = __fadd_rn(s, bd[j]);
}

// Many outputs (wide_rows_form and the like): one thread per output row and TB tokens.  A group of
// kDlAhead coalesced loads of the transposed weights is in flight while the group
// before is added; the tokens' inputs are the same for every lane (scalar loads).
// No LDS traffic is spent on products, and the TB chains of a thread hide each
// other's adds.  GATEUP: a thread has a neuron's gate and up rows.
constexpr int kDlAhead = 16;
template <bool GATEUP, int TB>
__global__ __launch_bounds__(64) void dl_wide_rows_kernel(const DcRows a, int out_f) {
  constexpr int M = GATEUP ? 2 : 1;
  const int64_t at = min((int64_t)blockIdx.x * 64 + threadIdx.x, a.nrows - 1);
  const int64_t r = dc_row(a, at);
  const int64_t b0 = (int64_t)blockIdx.y * TB;
  const DcMat* mat = &a.m[GATEUP ? 0 : blockIdx.z];
  const float* __restrict__ wt[M];
#pragma unroll
  for (int m = 0; m < M; ++m) wt[m] = mat[m].w + r;
  const float* __restrict__ xr[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) xr[t] = a.x + min(b0 + t, a.batch - 1) * a.ldx;
  float s[M][TB];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int t = 0; t < TB; ++t) s[m][t] = -0.0f;
  const int n = a.in_f, full = n / kDlAhead * kDlAhead;
  float w0[M][kDlAhead], w1[M][kDlAhead];
  auto load = [&](float (&w)[M][kDlAhead], int j) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int u = 0; u < kDlAhead; ++u) w[m][u] = wt[m][(int64_t)min(j + u, n - 1) * out_f];
  };
  auto add = [&](const float (&w)[M][kDlAhead], int j) {
#pragma unroll
    for (int u = 0; u < kDlAhead; ++u)
#pragma unroll
      for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int m = 0; m < M; ++m) s[m][t] = __fadd_rn(s[m][t], __fmul_rn(w[m][u], xr[t][j + u]));
  };
  load(w0, 0);
  int j = 0;
  for (; j + 2 * kDlAhead <= full; j += 2 * kDlAhead) {
    load(w1, j + kDlAhead);
    __builtin_amdgcn_sched_barrier(0);
    add(w0, j);
    load(w0, j + 2 * kDlAhead);
    __builtin_amdgcn_sched_barrier(0);
    add(w1, j + kDlAhead);
  }
  if (j < full) {
    add(w0, j);
    j += kDlAhead;
  }
  for (; j < n; ++j)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float w = wt[m][(int64_t)j * out_f];
#pragma unroll
      for (int t = 0; t < TB; ++t) s[m][t] = __fadd_rn(s[m][t], __fmul_rn(w, xr[t][j]));
    }
  if ((int64_t)blockIdx.x * 64 + threadIdx.x >= a.nrows) return;
  float bi[M];
#pragma unroll
  for (int m = 0; m < M; ++m) bi[m] = mat[m].bias[r];
#pragma unroll
  for (int t = 0; t < TB; ++t)
    if (b0 + t < a.batch) {
      const float z = __fadd_rn(s[0][t], bi[0]);
      mat->y[(b0 + t) * a.ldy + (a.scatter ? r : at)] =
          GATEUP ? __fmul_rn(silu_ref(z), __fadd_rn(s[M - 1][t], bi[M - 1])) : z;
    }
}

// The down projection's: one thread per output column and TB tokens, the selected
// neurons' columns read as rows of the transposed weights.
template <int TB>
__global__ __launch_bounds__(64) void dl_wide_down_kernel(
    const float* __restrict__ wdt, const float* __restrict__ bd, int hidden,
    const float* __restrict__ h, int64_t batch, const int64_t* __restrict__ sel, int n,
    float* __restrict__ y) {
  const int j = min((int)blockIdx.x * 64 + (int)threadIdx.x, hidden - 1);
  const int64_t b0 = (int64_t)blockIdx.y * TB;
  const float* __restrict__ hr[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) hr[t] = h + min(b0 + t, batch - 1) * n;
  float s[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) s[t] = 0.0f;
  const int full = n / kDlAhead * kDlAhead;
  int id[kDlAhead];                              // neurons of the group to load next
  float w0[kDlAhead], w1[kDlAhead];
  auto ids = [&](int a0) {
#pragma unroll
    for (int u = 0; u < kDlAhead; ++u) id[u] = (int)sel[min(a0 + u, n - 1)];
  };
  auto load = [&](float (&w)[kDlAhead]) {
#pragma unroll
    for (int u = 0; u < kDlAhead; ++u) w[u] = wdt[(size_t)id[u] * hidden + j];
  };
  // a zero activation adds nothing, whatever the weight
  auto add = [&](const float (&w)[kDlAhead], int a0) {
#pragma unroll
    for (int u = 0; u < kDlAhead; ++u)
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const float v = hr[t][a0 + u];
        s[t] = __fadd_rn(s[t], v != 0.0f ? __fmul_rn(w[u], v) : -0.0f);
      }
  };
  auto add_some = [&](const float (&w)[kDlAhead], int a0) {
#pragma unroll
    for (int u = 0; u < kDlAhead; ++u)
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const float v = hr[t][min(a0 + u, n - 1)];
        s[t] = __fadd_rn(s[t], a0 + u < n && v != 0.0f ? __fmul_rn(w[u], v) : -0.0f);
      }
  };
  if (n > 0) {
    ids(0);
    load(w0);
    ids(kDlAhead);
    int a0 = 0;
    for (; a0 + 2 * kDlAhead <= full; a0 += 2 * kDlAhead) {
      load(w1);
      ids(a0 + 2 * kDlAhead);
      __builtin_amdgcn_sched_barrier(0);
      add(w0, a0);
      load(w0);
      ids(a0 + 3 * kDlAhead);
      __builtin_amdgcn_sched_barrier(0);
      add(w1, a0 + kDlAhead);
    }
    if (a0 < n) {
      if (a0 + kDlAhead < n) load(w1);
      add_some(w0, a0);
      if (a0 + kDlAhead < n) add_some(w1, a0 + kDlAhead);
    }
  }
  if ((int)blockIdx.x * 64 + (int)threadIdx.x >= hidden) return;
  const float bi = bd[j];
#pragma unroll
  for (int t = 0; t < TB; ++t)
    if (b0 + t < batch) y[(b0 + t) * hidden + j] = __fadd_rn(s[t], bi);
}

// One wave per (head, token): the score's products in LDS, added by one lane in
// order, then the scaled v; zeros for a head that is not selected (att rows are
// whole).  q, k, v, att: [batch][qd].
constexpr int kDlHeadTile = 64;
__global__ __launch_bounds__(64) void dl_head_score_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    float* __restrict__ att, int64_t qd, int head_dim, const int64_t* __restrict__ heads,
    int64_t n_heads, float scale) {
  __shared__ float4 p4[kDlHeadTile / 4];
  float* p = reinterpret_cast<float*>(p4);
  const int lane = threadIdx.x;
  const int64_t head = blockIdx.x;
  const int64_t st = (int64_t)blockIdx.y * qd + head * head_dim;
  bool on = false;
  for (int64_t i = lane; i < n_heads; i += 64) on = on || heads[i] == head;
  if (__ballot(on) == 0ull) {
    for (int d = lane; d < head_dim; d += 64) att[st + d] = 0.0f;
    return;
  }
  float s = -0.0f;
  for (int d0 = 0; d0 < head_dim; d0 += kDlHeadTile) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kDlHeadTile / 64; ++u) {
      const int d = d0 + u * 64 + lane;
      const int64_t at = st + min(d, head_dim - 1);
      const float pr = __fmul_rn(q[at], k[at]);
      p[u * 64 + lane] = d < head_dim ? pr : -0.0f;
    }
    __syncthreads();
    s = chain_add_static<kDlHeadTile / 4, 1>(p4, s);   // every lane: the same sum
  }
  const float sc = sigmoid_ref(__fdiv_rn(s, scale));
  for (int d = lane; d < head_dim; d += 64) att[st + d] = __fmul_rn(v[st + d], sc);
}

// Lists of up to kDlArgList indices travel in the launch itself: the caller's
// list may be freed on return and nothing waits, where a copy from pageable host
// memory made every call wait for its stream (SparseMlp with 822 neurons, then
// SparseAttention with 6 heads, 3 tokens: 61.8 -> 40.9 us).  Longer lists are copied.
constexpr int kDlArgList = 960;
struct DlList {
  int32_t v[kDlArgList];
};
__global__ __launch_bounds__(kDlThreads) void dl_list_kernel(const DlList l, int n, int64_t* __restrict__ out) {
  for (int i = threadIdx.x; i < n; i += kDlThreads) out[i] = l.v[i];
}

// Checks idx_host[0..n) against [0, bound) and puts it into slot 0 of the
// stream's workspace w.
static int upload_indices(WsSet* w, const int64_t* idx_host, int64_t n, int64_t bound,
                          const char* what, hipStream_t st, const int64_t** out) {
  for (int64_t a = 0; a < n; ++a)
    KH_CHECK_ARG(idx_host[a] >= 0 && idx_host[a] < bound,
                 "%s index %lld out of range (%lld)", what, (long long)idx_host[a],
                 (long long)bound);
  int64_t* d = static_cast<int64_t*>(w->get(0, sizeof(int64_t) * (size_t)(n > 0 ? n : 1)));
  if (!d) return KH_ERR_ALLOC;
  if (n > 0 && n <= kDlArgList) {
    DlList l;
    for (int64_t a = 0; a < n; ++a) l.v[a] = static_cast<int32_t>(idx_host[a]);   // bound is an int
    hipLaunchKernelGGL(dl_list_kernel, dim3(1), dim3(kDlThreads), 0, st, l, (int)n, d);
    KH_LAUNCHED();
  } else if (n > 0) {
    KH_HIP(hipMemcpyAsync(d, idx_host, sizeof(int64_t) * (size_t)n, hipMemcpyHostToDevice, st));
    KH_HIP(hipStreamSynchronize(st));
  }
  *out = d;
  return KH_OK;
}

// Which form a call takes.  A chain block costs 3.5 to 4 us and 6 ns a term, whatever part of
// it is used, and kDcRound outputs' blocks run at once; the wide forms cost a term more but
// take many times as many outputs in that time.  `outputs`: in whole chain blocks.
constexpr int64_t kDcRound = 1 << 15;
// Rows of a Linear, us on the device, chains / wide.  32 inputs: 16384 outputs 5.9 / 3.3, 262144
// 69 / 4.1; 96: 1024 outputs 4.2 / 4.2, 16384 5.9 / 4.8; 128: 4096 of one token 4.4 / 4.9; 256: 16384
// 5.9 / 8.9, 65536 18.9 / 9.4; 512: 65536 20.5 / 16.6; 1024: 65536 28.0 / 30.4, 131072 55 / 30, 262144
// 107 / 36; 2048: 65536 43 / 58, 262144 168 / 68.
static bool wide_rows_form(int64_t outputs, int64_t terms) {
  return terms <= 96 || outputs > (terms <= 512 ? 1 : 3) * kDcRound;
}
// Gate and up rows of n of `of` neurons (two outputs a neuron).  Few of many leave a lane alone on its
// line of the transposed rows, which counts the more the longer they are.  64 inputs: wide is the
// faster at any size; 128 inputs, 30 of 2752: 64 tokens 2 us slower, 1024 5 faster; 256 inputs, 200 of
// 2752: 256 tokens 3 us faster, 4096 322 faster, 30 of 2752: 4096 7 slower; 512 inputs, 800 of 2752: 64
// tokens 2 us faster, 256 58 faster, 200 of 2752: 1024 60 slower; 1024 inputs, 800 of 2752: 64 tokens
// 15 us slower, 256 38 faster.
static bool wide_gateup_form(int64_t outputs, int64_t terms, int64_t n, int64_t of) {
  return terms <= 96 ||
         (outputs > kDcRound && 160 * outputs > terms * kDcRound && (terms <= 128 || n * 4096 >= of * terms));
}
// The down projection over n neurons, whose columns it gathers: 90 ns a term.  8 neurons: 16384 outputs
// the same, 32768 4 us faster; 30: 16384 4 us slower, 65536 6 faster; 200: 65536 5 us slower, 131072 8
// faster; 800: 131072 25 us slower, 262144 16 faster.
static bool wide_down_form(int64_t outputs, int64_t n) { return 160 * outputs > (128 + n) * kDcRound; }
// Waves of one token each below which a thread takes two tokens rather than four
// (1024: 256 tokens 35.4 with two, 38.2 with four; 1024 tokens 96.9, 69.5).
constexpr int64_t kDlWideSplit = 6144;

template <bool GATEUP, int TB>
static void chain_rows_go(const DcRows& a, bool vec, int mats, hipStream_t st) {
  const int own = GATEUP ? kDcRows / 2 : kDcRows;
  const dim3 g((unsigned)ceil_div(a.nrows, own), (unsigned)ceil_div(a.batch, TB), (unsigned)mats);
  if (vec)
    hipLaunchKernelGGL((dl_chain_rows_kernel<GATEUP, TB, true>), g, dim3(kDcThreads), 0, st, a);
  else
    hipLaunchKernelGGL((dl_chain_rows_kernel<GATEUP, TB, false>), g, dim3(kDcThreads), 0, st, a);
}

// Tokens per block: no more than the batch needs (a token's chains cost LDS).
template <bool GATEUP>
static int chain_rows(DcRows a, int mats, hipStream_t st) {
  const bool vec = a.in_f % 4 == 0 && a.ldx % 4 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0;
  constexpr int64_t kMaxTokens = 65535;   // grid.y blocks of at least one token
  const float* x = a.x;
  const int64_t batch = a.batch;
  float* y[3] = {a.m[0].y, a.m[1].y, a.m[2].y};
  for (int64_t b0 = 0; b0 < batch; b0 += kMaxTokens) {
    a.batch = std::min(batch - b0, kMaxTokens);
    a.x = x + b0 * a.ldx;
    for (int i = 0; i < 3; ++i) a.m[i].y = y[i] ? y[i] + b0 * a.ldy : nullptr;
    if (a.batch == 1) chain_rows_go<GATEUP, 1>(a, vec, mats, st);
    else if (a.batch == 2) chain_rows_go<GATEUP, 2>(a, vec, mats, st);
    else chain_rows_go<GATEUP, 4>(a, vec, mats, st);
    KH_LAUNCHED();
  }
  return KH_OK;
}

template <bool GATEUP>
static int wide_rows(DcRows a, int out_f, int mats, hipStream_t st) {
  constexpr int64_t kMaxTokens = 65535 * 4;
  const float* x = a.x;
  const int64_t batch = a.batch;
  float* y[3] = {a.m[0].y, a.m[1].y, a.m[2].y};
  for (int64_t b0 = 0; b0 < batch; b0 += kMaxTokens) {
    a.batch = std::min(batch - b0, kMaxTokens);
    a.x = x + b0 * a.ldx;
    for (int i = 0; i < 3; ++i) a.m[i].y = y[i] ? y[i] + b0 * a.ldy : nullptr;
    const unsigned gx = (unsigned)ceil_div(a.nrows, 64);
    if (a.batch == 1)
      hipLaunchKernelGGL((dl_wide_rows_kernel<GATEUP, 1>), dim3(gx, 1, (unsigned)mats), dim3(64), 0, st, a, out_f);
    else if (a.batch < 4 || (int64_t)gx * a.batch * mats < kDlWideSplit)
      hipLaunchKernelGGL((dl_wide_rows_kernel<GATEUP, 2>), dim3(gx, (unsigned)ceil_div(a.batch, 2), (unsigned)mats), dim3(64), 0,
                         st, a, out_f);
    else
      hipLaunchKernelGGL((dl_wide_rows_kernel<GATEUP, 4>), dim3(gx, (unsigned)ceil_div(a.batch, 4), (unsigned)mats), dim3(64), 0,
                         st, a, out_f);
    KH_LAUNCHED();
  }
  return KH_OK;
}

// `mats` projections of one shape (bias, outputs y[i]) of the same inputs.
static int rows_launch(const kh_dejavu_linear* const* l, int mats, const float* x, int64_t ldx,
                       int64_t batch, const int64_t* rows, int64_t nrows, float* const* y,
                       int64_t ldy, int scatter, int head_dim, hipStream_t st) {
  if (batch * nrows == 0) return KH_OK;
  const bool wide = wide_rows_form(mats * batch * ceil_div(nrows, kDcRows) * kDcRows, l[0]->in_f);
  DcRows a{};
  for (int i = 0; i < mats; ++i) a.m[i] = {wide ? l[i]->wt : l[i]->w, l[i]->bias, y[i]};
  a.in_f = l[0]->in_f;
  a.x = x;
  a.ldx = ldx;
  a.batch = batch;
  a.rows = rows;
  a.nrows = nrows;
  a.ldy = ldy;
  a.scatter = scatter;
  a.head_dim = head_dim;
  if (wide) return wide_rows<false>(a, l[0]->out_f, mats, st);
  return chain_rows<false>(a, mats, st);
}

template <int TB>
static void down_go(const kh_dejavu_linear* d, bool wide, const float* h, int64_t batch, const int64_t* sel,
                    int n, float* y, hipStream_t st) {
  const int H = d->out_f;
  const dim3 g((unsigned)ceil_div(H, wide ? 64 : kDcRows), (unsigned)ceil_div(batch, TB));
  if (wide)
    hipLaunchKernelGGL(dl_wide_down_kernel<TB>, g, dim3(64), 0, st, d->wt, d->bias, H, h, batch, sel, n, y);
  else if (H % 4 == 0)
    hipLaunchKernelGGL((dl_chain_down_kernel<TB, true>), g, dim3(kDcThreads), 0, st, d->wt, d->bias, H, h, batch,
                       sel, n, y);
  else
    hipLaunchKernelGGL((dl_chain_down_kernel<TB, false>), g, dim3(kDcThreads), 0, st, d->wt, d->bias, H, h, batch,
                       sel, n, y);
}

}  // namespace kh

using namespace kh;

extern "C" int kh_dejavu_linear_create(int in_features, int out_features, const float* w_host,
                                       const float* b_host, kh_dejavu_linear** out) {
  KH_CHECK_ARG(out && w_host && b_host, "null argument");
  KH_CHECK_ARG(in_features > 0 && out_features > 0, "bad shape (in %d out %d)", in_features,
               out_features);
  *out = nullptr;
  const size_t n = (size_t)in_features * (size_t)out_features;
  auto* l = new kh_dejavu_linear;
  l->in_f = in_features;
  l->out_f = out_features;
  l->w = static_cast<float*>(dev_alloc(n * sizeof(float)));
  l->wt = static_cast<float*>(dev_alloc(n * sizeof(float)));
  l->bias = static_cast<float*>(dev_alloc((size_t)out_features * sizeof(float)));
  if (!l->w || !l->wt || !l->bias) {
    kh_dejavu_linear_destroy(l);
    return KH_ERR_ALLOC;
  }
  hipError_t e = hipMemcpy(l->w, w_host, n * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(l->bias, b_host, (size_t)out_features * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(transpose_kernel<float>, dim3(ceil_div(in_features, 32), ceil_div(out_features, 32)),
                       dim3(256), 0, 0, l->w, out_features, in_features, l->wt);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);   // other streams go on
  }
  if (e != hipSuccess) {
    set_error("linear upload failed: %s", hipGetErrorString(e));
    kh_dejavu_linear_destroy(l);
    return KH_ERR_HIP;
  }
  *out = l;
  return KH_OK;
}

extern "C" int kh_dejavu_linear_destroy(kh_dejavu_linear* l) {
  if (!l) return KH_OK;
  dev_free(l->w);
  dev_free(l->wt);
  dev_free(l->bias);
  delete l;
  return KH_OK;
}

extern "C" int kh_dejavu_linear_forward(const kh_dejavu_linear* l, const float* x_dev,
                                        int64_t batch, float* y_dev, void* stream) {
  KH_CHECK_ARG(l && x_dev && y_dev, "null argument");
  KH_CHECK_ARG(batch >= 0, "bad batch");
  return rows_launch(&l, 1, x_dev, l->in_f, batch, nullptr, l->out_f, &y_dev, l->out_f, 0, 0,
                     as_stream(stream));
}

extern "C" int kh_dejavu_linear_forward_sparse(const kh_dejavu_linear* l, const float* x_dev,
                                               int64_t batch, const int64_t* idx_host,
                                               int64_t n_idx, float* y_dev, void* stream) {
  KH_CHECK_ARG(l && x_dev && y_dev && (idx_host || n_idx == 0), "null argument");
  KH_CHECK_ARG(batch >= 0 && n_idx >= 0, "bad shape");
  if (batch * n_idx == 0) return KH_OK;
  hipStream_t st = as_stream(stream);
  const int64_t* rows = nullptr;
  int rc = upload_indices(l->ws.get(st), idx_host, n_idx, l->out_f, "row", st, &rows);
  if (rc != KH_OK) return rc;
  return rows_launch(&l, 1, x_dev, l->in_f, batch, rows, n_idx, &y_dev, n_idx, 0, 0, st);
}

extern "C" int kh_dejavu_sparse_mlp_create(int hidden, int inter, kh_dejavu_sparse_mlp** out) {
  KH_CHECK_ARG(out, "null argument");
  KH_CHECK_ARG(hidden > 0 && inter > 0, "bad shape");
  auto* m = new kh_dejavu_sparse_mlp;
  m->hidden = hidden;
  m->inter = inter;
  *out = m;
  return KH_OK;
}

extern "C" int kh_dejavu_sparse_mlp_destroy(kh_dejavu_sparse_mlp* m) {
  delete m;
  return KH_OK;
}

extern "C" int kh_dejavu_sparse_mlp_forward(const kh_dejavu_sparse_mlp* m, const float* x_dev,
                                            int64_t batch, const kh_dejavu_linear* gate,
                                            const kh_dejavu_linear* up,
                                            const kh_dejavu_linear* down, const int64_t* sel_host,
                                            int64_t n_sel, float* y_dev, void* stream) {
  KH_CHECK_ARG(m && gate && up && down && x_dev && y_dev && (sel_host || n_sel == 0),
               "null argument");
  KH_CHECK_ARG(batch >= 0 && n_sel >= 0, "bad shape");
  const int H = m->hidden, I = m->inter;
  KH_CHECK_ARG(gate->in_f == H && gate->out_f == I && up->in_f == H && up->out_f == I &&
                   down->in_f == I && down->out_f == H,
               "projection shapes do not match hidden %d / intermediate %d", H, I);
  if (batch == 0) return KH_OK;
  hipStream_t st = as_stream(stream);
  const int64_t* sel = nullptr;
  int rc = upload_indices(m->ws.get(st), sel_host, n_sel, I, "neuron", st, &sel);
  if (rc != KH_OK) return rc;
  float* h = static_cast<float*>(m->ws.get(st)->get(1, sizeof(float) * (size_t)(batch * n_sel + 1)));
  if (!h) return KH_ERR_ALLOC;
  if (batch * n_sel > 0) {
    DcRows g{};
    const bool wide = wide_gateup_form(batch * ceil_div(n_sel, kDcRows / 2) * kDcRows, H, n_sel, I);
    g.m[0] = {wide ? gate->wt : gate->w, gate->bias, h};
    g.m[1] = {wide ? up->wt : up->w, up->bias, nullptr};
    g.in_f = H;
    g.x = x_dev;
    g.ldx = H;
    g.batch = batch;
    g.rows = sel;
    g.nrows = n_sel;
    g.ldy = n_sel;
    rc = wide ? wide_rows<true>(g, I, 1, st) : chain_rows<true>(g, 1, st);
    if (rc != KH_OK) return rc;
  }
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    const int64_t nb = std::min<int64_t>(batch - b0, 65535);
    const float* hb = h + b0 * n_sel;
    float* yb = y_dev + b0 * H;
    const bool wide = wide_down_form(nb * ceil_div(H, kDcRows) * kDcRows, n_sel);
    if (nb == 1) down_go<1>(down, wide, hb, nb, sel, (int)n_sel, yb, st);
    else if (nb == 2) down_go<2>(down, wide, hb, nb, sel, (int)n_sel, yb, st);
    else down_go<4>(down, wide, hb, nb, sel, (int)n_sel, yb, st);
    KH_LAUNCHED();
  }
  return KH_OK;
}

extern "C" int kh_dejavu_sparse_attention_create(int hidden, int num_heads, int head_dim,
                                                 kh_dejavu_sparse_attention** out) {
  KH_CHECK_ARG(out, "null argument");
  KH_CHECK_ARG(hidden > 0 && num_heads > 0 && head_dim > 0, "bad shape");
  auto* a = new kh_dejavu_sparse_attention;
  a->hidden = hidden;
  a->num_heads = num_heads;
  a->head_dim = head_dim;
  *out = a;
  return KH_OK;
}

extern "C" int kh_dejavu_sparse_attention_destroy(kh_dejavu_sparse_attention* a) {
  delete a;
  return KH_OK;
}

extern "C" int kh_dejavu_sparse_attention_forward(
    const kh_dejavu_sparse_attention* a, const float* x_dev, int64_t batch, const kh_dejavu_linear* q,
    const kh_dejavu_linear* k, const kh_dejavu_linear* v, const kh_dejavu_linear* o,
    const int64_t* heads_host, int64_t n_heads, float* y_dev, void* stream) {
  KH_CHECK_ARG(a && q && k && v && o && x_dev && y_dev && (heads_host || n_heads == 0),
               "null argument");
  KH_CHECK_ARG(batch >= 0 && n_heads >= 0, "bad shape");
  const int H = a->hidden, hd = a->head_dim;
  const int64_t qd = (int64_t)a->num_heads * hd;
  KH_CHECK_ARG(q->in_f == H && k->in_f == H && v->in_f == H && q->out_f == qd &&
                   k->out_f == qd && v->out_f == qd && o->in_f == qd && o->out_f == H,
               "projection shapes do not match hidden %d / %d heads x %d", H, a->num_heads, hd);
  if (batch == 0) return KH_OK;
  hipStream_t st = as_stream(stream);
  const int64_t* dl = nullptr;
  int rc = upload_indices(a->ws.get(st), heads_host, n_heads, a->num_heads, "head", st, &dl);
  if (rc != KH_OK) return rc;
  float* buf = static_cast<float*>(a->ws.get(st)->get(1, sizeof(float) * (size_t)(4 * batch * qd)));
  if (!buf) return KH_ERR_ALLOC;
  float *qv = buf, *kv = buf + batch * qd, *vv = buf + 2 * batch * qd, *att = buf + 3 * batch * qd;
  const kh_dejavu_linear* qkv[3] = {q, k, v};
  float* outs[3] = {qv, kv, vv};
  if ((rc = rows_launch(qkv, 3, x_dev, H, batch, dl, n_heads * hd, outs, qd, 1, hd, st)) != KH_OK) return rc;
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    const int64_t o0 = b0 * qd;
    hipLaunchKernelGGL(dl_head_score_kernel, dim3((unsigned)a->num_heads, (unsigned)std::min<int64_t>(batch - b0, 65535)),
                       dim3(64), 0, st, qv + o0, kv + o0, vv + o0, att + o0, qd, hd, dl, n_heads, sqrtf((float)hd));
    KH_LAUNCHED();
  }
  return rows_launch(&o, 1, att, qd, batch, nullptr, H, &y_dev, H, 0, 0, st);
}
