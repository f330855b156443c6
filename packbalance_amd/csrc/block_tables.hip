// Document block tables for packed sequences, for gfx950.
//
// Reference semantics: packbalance/model/attention.py:25-54 builds a
// FlexAttention BlockMask from the mask
//     allowed(q, kv) = doc[q] == doc[kv] && q >= kv
// through torch's create_block_mask, which materialises the dense
// [B, H, S, S] boolean mask, pads it with False to a multiple of the block
// size, sums each block and classifies it EMPTY / PARTIAL / FULL, then orders
// every row with argsort(descending, stable).
//
// Here the mask is never materialised.  One launch (block_table_rows) builds
// the eight int32 tables: a workgroup per (row, orientation, batch) classifies
// its row's tiles from the documents' runs (doc_tiles.hpp) and writes the row's
// four table rows for every head, set indices ascending then unset indices
// ascending -- the exact order of a stable descending argsort of a 0/1 row --
// with a ballot rank per tile.
//
// Rows of more tiles than fit in LDS take two launches: classify_tiles writes
// the class of every (q-block, kv-block) tile, from doc_ids staged in LDS, to the
// workspace, and order_tables turns a row of them into table rows, one thread
// per (batch, head, row).
#include "common.hpp"
#include "doc_tiles.hpp"

namespace pb {
namespace {

enum : uint8_t { kEmpty = kTileEmpty, kPartial = kTilePartial, kFull = kTileFull, kCausal = kTileCausal };

// The eight tables of one orientation pair: [0] by query block, [1] by KV block.
struct Tables {
  int32_t *num[2], *idx[2], *fnum[2], *fidx[2];
};

// grid = (2 * nblk, b): row r < nblk is query block r, else KV block r - nblk.
// A row's order is computed once (set tiles ascending, then the others: the
// tile's rank by ballot) and written for every head, one wave per head in
// turn.  Latency-bound (2 MB of tables at S 8192, 32 heads); in place of one
// wave per tile over all its pairs and one thread per table row (S 8192, 32
// heads): 66 -> 13 us.
__global__ __launch_bounds__(kTileThreads) void block_table_rows(const int64_t *__restrict__ doc,
                                                                 int64_t doc_stride, int64_t s,
                                                                 int block, int nblk, int nh,
                                                                 Tables t) {
  __shared__ OwnRuns runs;
  extern __shared__ uint8_t cls[];  // [nblk]
  const int b = blockIdx.y, o = (int)blockIdx.x >= nblk ? 1 : 0;
  const int r = (int)blockIdx.x - o * nblk;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  classify_row(runs, cls, doc + (int64_t)b * doc_stride, s, (int64_t)r * block, block, block, nblk,
               o != 0, false);
  __syncthreads();
  int np = 0, nf = 0;  // set tiles of the partial and the full table
  for (int c0 = 0; c0 < nblk; c0 += 64) {
    const uint8_t k = c0 + lane < nblk ? cls[c0 + lane] : kEmpty;
    np += __builtin_popcountll(__builtin_amdgcn_ballot_w64(k == kPartial));
    nf += __builtin_popcountll(__builtin_amdgcn_ballot_w64(k == kFull));
  }
  int sp = 0, sf = 0;  // set tiles before column block c0
  const uint64_t below = (1ull << lane) - 1ull;
  for (int c0 = 0; c0 < nblk; c0 += 64) {
    const int c = c0 + lane;
    const uint8_t k = c < nblk ? cls[c] : kEmpty;
    const uint64_t bp = __builtin_amdgcn_ballot_w64(k == kPartial);
    const uint64_t bf = __builtin_amdgcn_ballot_w64(k == kFull);
    const int rp = sp + __builtin_popcountll(bp & below), rf = sf + __builtin_popcountll(bf & below);
    if (c < nblk) {
      const int pp = k == kPartial ? rp : np + (c - rp), pf = k == kFull ? rf : nf + (c - rf);
      for (int h = wave; h < nh; h += kTileWaves) {
        const int64_t row = (((int64_t)b * nh + h) * nblk + r) * nblk;
        t.idx[o][row + pp] = c;
        t.fidx[o][row + pf] = c;
      }
    }
    sp += __builtin_popcountll(bp);
    sf += __builtin_popcountll(bf);
  }
  for (int h = threadIdx.x; h < nh; h += kTileThreads) {
    const int64_t row = ((int64_t)b * nh + h) * nblk + r;
    t.num[o][row] = np;
    t.fnum[o][row] = nf;
  }
}

// grid = (ceil(nkv / 4), nq, b); block = 256 threads, one wave per tile
// (kv tile 4 * blockIdx.x + wave).  qb x kb tile sizes in tokens.  The q
// documents of the row sit in LDS (read as broadcasts), lane j takes kv
// columns j, j + 64, ... and the three tile flags are wave ballots.
// With causal_class, a partial tile in which every in-range pair with kv <= q
// shares a document is reported as kCausal (its mask is the causal test).
__global__ __launch_bounds__(256) void classify_tiles(const int64_t *__restrict__ doc,
                                                      int64_t doc_stride, int64_t s, int qbs,
                                                      int kbs, int nq, int nkv, int causal_class,
                                                      uint8_t *__restrict__ cls) {
  extern __shared__ int64_t sdoc[];  // [qbs] q docs
  const int qb = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kb = blockIdx.x * 4 + wave;
  const int64_t q0 = (int64_t)qb * qbs, k0 = (int64_t)kb * kbs;
  const int64_t *drow = doc + (int64_t)b * doc_stride;
  for (int i = threadIdx.x; i < qbs; i += 256) sdoc[i] = (q0 + i < s) ? drow[q0 + i] : 0;
  __syncthreads();
  if (kb >= nkv) return;
  uint8_t *out = cls + ((int64_t)b * nq + qb) * nkv + kb;
  // Every kv in the tile lies after every q: masked by causality.
  if (k0 > q0 + qbs - 1) {
    if (lane == 0) *out = kEmpty;
    return;
  }
  bool any = false, all = true, one_doc = true;
  for (int j = lane; j < kbs; j += 64) {
    const int64_t kv = k0 + j;
    const bool kin = kv < s;
    const int64_t dk = kin ? drow[kv] : 0;
    for (int i = 0; i < qbs; ++i) {
      const int64_t q = q0 + i;
      const bool causal = kin && q < s && q >= kv;
      const bool same = sdoc[i] == dk;
      any |= causal & same;
      all &= causal & same;
      one_doc &= !causal | same;
    }
  }
  const bool a_any = __builtin_amdgcn_ballot_w64(any) != 0;
  const bool a_all = __builtin_amdgcn_ballot_w64(!all) == 0;
  const bool a_one = __builtin_amdgcn_ballot_w64(!one_doc) == 0;
  if (lane == 0)
    *out = a_all ? kFull : !a_any ? kEmpty : (causal_class && a_one) ? kCausal : kPartial;
}

// One thread per (b, h, row) of either orientation.
//   rows [0, nq)        -> kv tables (row = q-block, scan over kv-blocks)
//   rows [nq, nq + nkv) -> q tables  (row = kv-block, scan over q-blocks)
__global__ __launch_bounds__(256) void order_tables(const uint8_t *__restrict__ cls, int nb, int nh,
                                                    int nq, int nkv, int32_t *kv_num,
                                                    int32_t *kv_idx, int32_t *fkv_num,
                                                    int32_t *fkv_idx, int32_t *q_num,
                                                    int32_t *q_idx, int32_t *fq_num,
                                                    int32_t *fq_idx) {
  const int64_t tid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per_bh = nq + nkv;
  if (tid >= (int64_t)nb * nh * per_bh) return;
  const int b = (int)(tid / ((int64_t)nh * per_bh));
  const int64_t rem = tid - (int64_t)b * nh * per_bh;
  const int h = (int)(rem / per_bh);
  const int r = (int)(rem - (int64_t)h * per_bh);
  const uint8_t *C = cls + (int64_t)b * nq * nkv;
  const int64_t bh = (int64_t)b * nh + h;
  if (r < nq) {
    // kv-major tables for q-block r.
    const int qb = r;
    int32_t *pi = kv_idx + (bh * nq + qb) * nkv;
    int32_t *fi = fkv_idx + (bh * nq + qb) * nkv;
    int np = 0, nf = 0;
    for (int k = 0; k < nkv; ++k) {
      const uint8_t c = C[(int64_t)qb * nkv + k];
      if (c == kPartial) pi[np++] = k;
      if (c == kFull) fi[nf++] = k;
    }
    int tp = np, tf = nf;
    for (int k = 0; k < nkv; ++k) {
      const uint8_t c = C[(int64_t)qb * nkv + k];
      if (c != kPartial) pi[tp++] = k;
      if (c != kFull) fi[tf++] = k;
    }
    kv_num[bh * nq + qb] = np;
    fkv_num[bh * nq + qb] = nf;
  } else {
    const int kb = r - nq;
    int32_t *pi = q_idx + (bh * nkv + kb) * nq;
    int32_t *fi = fq_idx + (bh * nkv + kb) * nq;
    int np = 0, nf = 0;
    for (int q = 0; q < nq; ++q) {
      const uint8_t c = C[(int64_t)q * nkv + kb];
      if (c == kPartial) pi[np++] = q;
      if (c == kFull) fi[nf++] = q;
    }
    int tp = np, tf = nf;
    for (int q = 0; q < nq; ++q) {
      const uint8_t c = C[(int64_t)q * nkv + kb];
      if (c != kPartial) pi[tp++] = q;
      if (c != kFull) fi[tf++] = q;
    }
    q_num[bh * nkv + kb] = np;
    fq_num[bh * nkv + kb] = nf;
  }
}

}  // namespace

// Shared with the attention planner: classify tiles of qbs x kbs tokens.
int classify_doc_tiles(const int64_t *doc, int64_t doc_stride, int64_t b, int64_t s, int qbs,
                       int kbs, int causal_class, uint8_t *cls, hipStream_t st) {
  const int nq = (int)((s + qbs - 1) / qbs), nkv = (int)((s + kbs - 1) / kbs);
  dim3 grid((unsigned)((nkv + 3) / 4), nq, (unsigned)b);
  const size_t lds = (size_t)qbs * sizeof(int64_t);
  hipLaunchKernelGGL(classify_tiles, grid, dim3(256), lds, st, doc, doc_stride, s, qbs, kbs, nq, nkv,
                     causal_class, cls);
  return launch_status("classify_doc_tiles");
}

}  // namespace pb

extern "C" int pb_doc_block_tables(const int64_t *doc_ids, int64_t doc_stride, int64_t b,
                                   int64_t s, int64_t block, int64_t h, int32_t *kv_num,
                                   int32_t *kv_idx, int32_t *full_kv_num, int32_t *full_kv_idx,
                                   int32_t *q_num, int32_t *q_idx, int32_t *full_q_num,
                                   int32_t *full_q_idx, uint8_t *class_ws, void *stream) {
  using namespace pb;
  clear_error();
  PB_CHECK_ARG(b >= 1 && s >= 1 && h >= 1, "pb_doc_block_tables: bad shape b=%lld s=%lld h=%lld",
               (long long)b, (long long)s, (long long)h);
  PB_CHECK_ARG(block >= 1 && block <= 1024, "pb_doc_block_tables: block size %lld out of [1, 1024]",
               (long long)block);
  PB_CHECK_ARG(doc_stride >= s, "pb_doc_block_tables: doc_stride < s");
  const int64_t nblk = (s + block - 1) / block;
  PB_CHECK_SUPPORTED(nblk <= 65535 && b <= 65535, "pb_doc_block_tables: too many blocks");
  hipStream_t st = as_stream(stream);
  if (nblk <= kMaxRowTiles) {
    Tables t;
    t.num[0] = kv_num; t.idx[0] = kv_idx; t.fnum[0] = full_kv_num; t.fidx[0] = full_kv_idx;
    t.num[1] = q_num; t.idx[1] = q_idx; t.fnum[1] = full_q_num; t.fidx[1] = full_q_idx;
    hipLaunchKernelGGL(block_table_rows, dim3((unsigned)(2 * nblk), (unsigned)b), dim3(kTileThreads),
                       (size_t)nblk, st, doc_ids, doc_stride, s, (int)block, (int)nblk, (int)h, t);
    return launch_status("pb_doc_block_tables");
  }
  int rc = classify_doc_tiles(doc_ids, doc_stride, b, s, (int)block, (int)block, 0, class_ws, st);
  if (rc) return rc;
  const int64_t threads = b * h * (2 * nblk);
  hipLaunchKernelGGL(order_tables, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st,
                     class_ws, (int)b, (int)h, (int)nblk, (int)nblk, kv_num, kv_idx, full_kv_num,
                     full_kv_idx, q_num, q_idx, full_q_num, full_q_idx);
  return launch_status("pb_doc_block_tables");
}
