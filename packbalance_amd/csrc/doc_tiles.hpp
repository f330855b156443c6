// Classes of one row of document-mask tiles, by a workgroup (256 threads).
//
// The mask is allowed(q, kv) = doc[q] == doc[kv] && q >= kv.  A row is one tile
// of one axis (the row's "own" tile: queries, or KV positions when by_kv)
// against every tile of the other axis.  The own tile's documents are first
// reduced to runs of equal ids: against a run, a position of the other axis
// allows a pair, or every pair, depending only on its id and on which side of
// the run's bound it lies -- the run's last query, or its first KV position --
// so a tile costs (positions) x (runs) compares instead of (positions)^2, with
// the same answer for any ids, also ids that recur.  A run needs no order, so
// threads append them as they find them.
#pragma once

#include "common.hpp"

namespace pb {

enum : uint8_t { kTileEmpty = 0, kTilePartial = 1, kTileFull = 2, kTileCausal = 3 };

constexpr int kTileThreads = 256, kTileWaves = kTileThreads / 64;
constexpr int kMaxOwn = 1024;         // own tile length
constexpr int64_t kMaxRowTiles = 16384;  // tiles of a row whose classes fit in LDS

struct OwnRuns {
  int64_t doc[kMaxOwn];
  int bound[kMaxOwn];
  int n;
};

// Fills cls[0 .. ncols) with the row's classes; the caller's barrier makes
// them visible.  own0 / own: first position and length of the own tile,
// other: length of the other axis' tiles.
__device__ __forceinline__ void classify_row(OwnRuns &runs, uint8_t *cls, const int64_t *doc,
                                             int64_t s, int64_t own0, int own, int other,
                                             int ncols, bool by_kv, bool causal_class) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t own_end = own0 + own < s ? own0 + own : s;  // in-range part
  if (tid == 0) runs.n = 0;
  __syncthreads();
  for (int64_t p = own0 + tid; p < own_end; p += kTileThreads) {
    const int64_t d = doc[p];
    const bool edge = by_kv ? p == own0 || doc[p - 1] != d : p + 1 == own_end || doc[p + 1] != d;
    if (edge) {
      const int i = atomicAdd(&runs.n, 1);
      runs.doc[i] = d;
      runs.bound[i] = (int)p;
    }
  }
  __syncthreads();
  const int n = runs.n;
  // Every pair allowed: one run, the whole own tile in range, and the other
  // positions all past (queries) or before (KV) it.
  const bool whole = n == 1 && own0 + own <= s;
  const int64_t far = by_kv ? own0 + own - 1 : own0;
  auto load = [&](int c) {
    const int64_t p = (int64_t)c * other + lane;
    return c < ncols && lane < other && p < s ? doc[p] : 0;
  };
  int64_t first = load(wave);
  for (int c = wave; c < ncols; c += kTileWaves) {
    const int64_t p0 = (int64_t)c * other;
    const int64_t next = load(c + kTileWaves);
    // Every kv lies after every q: masked by causality.
    const bool never = by_kv ? own0 > p0 + other - 1 : p0 > own0 + own - 1;
    uint8_t k = kTileEmpty;
    if (!never) {
      bool any = false, all = whole, one = true;
      for (int j = lane; j < other; j += 64) {
        const int64_t p = p0 + j;
        const bool in = p < s;
        const int64_t d = j < 64 ? first : in ? doc[p] : 0;
        for (int r = 0; r < n; ++r) {
          const bool side = in && (by_kv ? p >= runs.bound[r] : p <= runs.bound[r]);
          const bool same = d == runs.doc[r];
          any |= side & same;
          one &= !side | same;
        }
        all &= in && d == runs.doc[0] && (by_kv ? p >= far : p <= far);
      }
      if (__builtin_amdgcn_ballot_w64(!all) == 0) k = kTileFull;
      else if (__builtin_amdgcn_ballot_w64(any) != 0)
        k = causal_class && __builtin_amdgcn_ballot_w64(!one) == 0 ? kTileCausal : kTilePartial;
    }
    if (lane == 0) cls[c] = k;
    first = next;
  }
}

}  // namespace pb
