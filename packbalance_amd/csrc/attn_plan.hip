// Tile plans for the document-masked attention kernels.
//
// A plan lists, for every row tile of one orientation, the non-empty tiles of
// the other orientation in ascending order, each tagged FULL (no element mask
// needed), CAUSAL (one document for every pair with kv <= q: the causal test
// is the whole mask) or PARTIAL.  It is the attention kernels' form of the FlexAttention
// block tables (kv_indices / full_kv_indices for by_kv = 0, q_indices /
// full_q_indices for by_kv = 1), at the kernels' own tile sizes, with FULL and
// PARTIAL merged into one ascending list so a kernel walks one array.
#include "attn_common.hpp"
#include "doc_tiles.hpp"

namespace pb {
namespace {

enum : uint8_t { kEmpty = kTileEmpty, kPartial = kTilePartial, kFull = kTileFull, kCausal = kTileCausal };

// The set tiles of a row of classes C (column stride cs), in order, by one
// wave: 64 columns at a time, each lane's rank among the set lanes below it.
__device__ __forceinline__ void compact_row(const uint8_t *C, int64_t cs, int ncols, int lane,
                                            int32_t *L, int32_t *count) {
  int n = 0;
  for (int c0 = 0; c0 < ncols; c0 += 64) {
    const int c = c0 + lane;
    const uint8_t v = c < ncols ? C[c * cs] : kEmpty;
    const uint64_t set = __builtin_amdgcn_ballot_w64(v != kEmpty);
    if (v != kEmpty) {
      const int rank = __builtin_popcountll(set & ((1ull << lane) - 1ull));
      L[n + rank] = (c << 2) | (v == kFull ? 1 : v == kCausal ? 2 : 0);
    }
    n += __builtin_popcountll(set);
  }
  if (lane == 0) *count = n;
}

// A workgroup per plan row: the row's classes from the documents' runs
// (doc_tiles.hpp), then its list.  Latency-bound.  In place of a launch over
// all tiles' pairs and one over the rows: [8, 8192] at 128 x 64, 188 + 4 -> 25 us.
__global__ __launch_bounds__(kTileThreads) void plan_rows(const int64_t *__restrict__ doc,
                                                          int64_t doc_stride, int64_t s, int own,
                                                          int other, int nrows, int ncols,
                                                          int by_kv, int32_t *__restrict__ counts,
                                                          int32_t *__restrict__ lists) {
  __shared__ OwnRuns runs;
  extern __shared__ uint8_t cls[];  // [ncols]
  const int r = blockIdx.x, b = blockIdx.y;
  classify_row(runs, cls, doc + (int64_t)b * doc_stride, s, (int64_t)r * own, own, other, ncols,
               by_kv != 0, true);
  __syncthreads();
  if (threadIdx.x < 64) {
    const int64_t row = (int64_t)b * nrows + r;
    compact_row(cls, 1, ncols, threadIdx.x, lists + row * ncols, counts + row);
  }
}

// Rows of more tiles than fit in LDS: one wave per row of the class bytes that
// classify_doc_tiles left in the workspace.
__global__ __launch_bounds__(256) void plan_lists(const uint8_t *__restrict__ cls, int nb, int nq,
                                                  int nk, int by_kv, int32_t *__restrict__ counts,
                                                  int32_t *__restrict__ lists) {
  const int nrows = by_kv ? nk : nq, ncols = by_kv ? nq : nk;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= (int64_t)nb * nrows) return;
  const int b = (int)(row / nrows), r = (int)(row - (int64_t)b * nrows);
  const uint8_t *C = cls + (int64_t)b * nq * nk + (by_kv ? (int64_t)r : (int64_t)r * nk);
  compact_row(C, by_kv ? nk : 1, ncols, threadIdx.x & 63, lists + row * ncols, counts + row);
}

}  // namespace
}  // namespace pb

extern "C" int pb_attn_plan(const int64_t *doc_ids, int64_t doc_stride, int64_t b, int64_t s,
                            int64_t q_tile, int64_t kv_tile, int by_kv, int32_t *counts,
                            int32_t *lists, uint8_t *class_ws, void *stream) {
  using namespace pb;
  clear_error();
  PB_CHECK_ARG(b >= 1 && s >= 1, "pb_attn_plan: bad shape b=%lld s=%lld", (long long)b, (long long)s);
  PB_CHECK_ARG(q_tile >= 1 && q_tile <= 1024 && kv_tile >= 1 && kv_tile <= 1024,
               "pb_attn_plan: tile sizes out of [1, 1024]");
  PB_CHECK_ARG(doc_stride >= s, "pb_attn_plan: doc_stride < s");
  PB_CHECK_ARG(by_kv == 0 || by_kv == 1, "pb_attn_plan: by_kv must be 0 or 1");
  hipStream_t st = as_stream(stream);
  const int nq = (int)((s + q_tile - 1) / q_tile), nk = (int)((s + kv_tile - 1) / kv_tile);
  const int own = (int)(by_kv ? kv_tile : q_tile), other = (int)(by_kv ? q_tile : kv_tile);
  const int nrows = by_kv ? nk : nq, ncols = by_kv ? nq : nk;
  if (ncols <= kMaxRowTiles && b <= 65535) {
    hipLaunchKernelGGL(plan_rows, dim3((unsigned)nrows, (unsigned)b), dim3(kTileThreads),
                       (size_t)ncols, st, doc_ids, doc_stride, s, own, other, nrows, ncols, by_kv,
                       counts, lists);
    return launch_status("pb_attn_plan");
  }
  int rc = classify_doc_tiles(doc_ids, doc_stride, b, s, (int)q_tile, (int)kv_tile, 1, class_ws, st);
  if (rc) return rc;
  const int64_t rows = b * nrows;
  hipLaunchKernelGGL(plan_lists, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, class_ws,
                     (int)b, nq, nk, by_kv, counts, lists);
  return launch_status("pb_attn_plan");
}
