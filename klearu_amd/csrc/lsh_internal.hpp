// lsh_internal.hpp -- handle layouts shared by lsh.hip and slide.hip.
#pragma once
#include <vector>

#include "common.hpp"

struct kh_hash_family {
  int dim = 0, k = 0, L = 0;
  int kind = KH_FAMILY_TERNARY;          // KH_FAMILY_*: hyperplanes or a rank-based family
  int ws = 0, bits = 0;                  // WTA / DWTA: window size, bits per window
  std::vector<uint32_t> windows_host;    // WTA / DWTA [L][k][ws]
  uint32_t* windows_dev = nullptr;
  uint32_t* fallback_dev = nullptr;      // DWTA [L][k]: empty-window position
  std::vector<uint32_t> perms_host;      // MinHash [L][dim]
  uint32_t* perms_dev = nullptr;
  std::vector<int8_t> planes_host;  // [L][k][dim]
  // Nonzero lists of the planes, transposed so that the planes handled by
  // consecutive lanes are adjacent: entry j of plane p at ent_t[j*L*k + p],
  // (dim << 1) | (sign < 0), in dimension order; rows past a plane's nnz are 0.
  int32_t* nnz = nullptr;           // [L*k]
  uint32_t* ent_t = nullptr;        // [ent_rows][L*k]
  int ent_rows = 0;                 // max nnz rounded up to the hash kernel's batch
  // Planes as BF16 matrix-core operands (L*k <= 1024, dim <= 8192):
  // [ceil(dim/32)][ceil(L*k/16)][64 lanes] x 8 values; null otherwise.
  uint4* bt_dev = nullptr;
  int bt_ksteps = 0, bt_tiles = 0;
  // The same planes' 2-bit signs plane by plane, [L*k][ceil(dim/16)] words (01 = +1,
  // 11 = -1), for the sums the matrix cores leave undecided.
  uint32_t* sp_dev = nullptr;
  // 2-bit plane signs for the per-row kernels: group g holds tables g*sg_tpb.. (planes q = 0..sg_tpb*k-1 of the
  // group), as [dim][sg_words] words, plane q in bits 2(q%16), 2(q%16)+1 of
  // word q/16 (01 = +1, 11 = -1, 00 = no term); each group padded to sg_n4
  // uint4.  Null for the rank-based families.
  uint4* sg_dev = nullptr;
  int sg_tpb = 0, sg_groups = 0, sg_words = 0, sg_n4 = 0;
};

namespace kh {
// Grow-only device scratch slots of an index's mutation calls, used as a stack.
struct ScratchArena {
  std::vector<std::pair<void*, size_t>> slots;
  size_t cursor = 0;
  ScratchArena() = default;
  ScratchArena(const ScratchArena&) = delete;
  ScratchArena& operator=(const ScratchArena&) = delete;
  ~ScratchArena() {
    for (auto& s : slots) dev_free(s.first);
  }
};
}  // namespace kh

struct kh_lsh_index {
  const kh_hash_family* h = nullptr;
  int type = 0, cap = 0, L = 0, k = 0, nb = 0;
  uint32_t* data = nullptr;   // [L][nb][cap]
  uint32_t* len = nullptr;    // [L][nb]
  uint64_t* count = nullptr;  // [L][nb]
  uint32_t id_bound = 0;      // 1 + largest id inserted so far (ids are below 2^31)
  mutable kh::StreamWs ws;    // query scratch per stream
  kh::ScratchArena arena;     // insert / remove / rebuild scratch, kept between calls
  uint32_t* mx_host = nullptr;  // pinned: the largest id of an insert call
  hipEvent_t mx_done = nullptr; // recorded when it is written
};

namespace kh {

int hash_dense_launch(const kh_hash_family* h, const float* x, int64_t ldx, int64_t batch,
                      uint32_t* codes, hipStream_t st);
// Row r holds entries xoff[r * xstep] .. xoff[r * xstep + 1]: CSR offsets with
// xstep 1, one (start, end) pair per row with xstep 2.
int hash_sparse_launch(const kh_hash_family* h, const int64_t* xoff, const uint32_t* xidx,
                       const float* xval, int64_t batch, uint32_t* codes, hipStream_t st, int xstep = 1);
// Per-row unique ids (ascending) and hit counts into [batch][stride] buffers.
int query_launch(const kh_lsh_index* idx, const uint32_t* qcodes, int64_t batch, uint32_t* qids,
                 uint32_t* qcnt, int stride, int32_t* ulen, hipStream_t st);
int query_stride(const kh_lsh_index* idx);
// Whether short dense batches hash with their signs staged in LDS.
bool hash_dense_rows(const kh_hash_family* h);
// The rank-based families (hash_rank.hip), called by the two launchers above.
int rank_hash_dense_launch(const kh_hash_family* h, const float* x, int64_t ldx, int64_t batch,
                           uint32_t* codes, hipStream_t st);
int rank_hash_sparse_launch(const kh_hash_family* h, const int64_t* xoff, const uint32_t* xidx,
                            const float* xval, int64_t batch, uint32_t* codes, hipStream_t st, int xstep);
// Row lengths -> CSR offsets, copies of up to four per-row arrays, then a
// synchronising capacity check.
int csr_finish(const uint32_t* qids, const uint32_t* qcnt, const float* f1, const float* f2,
               int stride, const int32_t* ulen, int64_t batch, int64_t* off, uint32_t* ids,
               uint32_t* cnts, float* o1, float* o2, int64_t capacity, hipStream_t st);
// csr_finish's capacity check alone, for kernels that write CSR rows themselves.
int csr_check(const int64_t* off, int64_t batch, int stride, int64_t capacity, hipStream_t st);
// Rows of a batch up to which a block sums the lengths before its row itself.
constexpr int kCsrPackMax = 4096;

}  // namespace kh
