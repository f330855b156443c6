// Classes of one row of document-mask tiles, by a workgroup.
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
//
// An own tile of many short documents has many runs, and one wave compares them
// with tile after tile.  So the runs' ids also set bits of a hash table: a tile
// none of whose ids hits one is empty (most are, whatever the order of the ids),
// and the compares stop once the class is decided.  S 8192, captured launches in
// us, a wave for every tile over all its pairs / every run against every tile /
// sifted: the tables of one head, documents of one token 56 / 532 / 16, of about 5
// tokens 56 / 131 / 12, of 200 57 / 22 / 13; three plans (128 x 64, 64 x 64 twice) 84
// / 1118 / 35, 84 / 292 / 29, 84 / 78 / 47.  Eight waves: with four a short row of 32 x 32
// tiles (the plans of [1, 2048], 12 / 4 heads, D 64) took 28 us, now 18, with sixteen
// 13, but large grids longer ([100, 512] 12 / 15 / 29 us with 4 / 8 / 16).
#pragma once

#include "common.hpp"

namespace pb {

enum : uint8_t { kTileEmpty = 0, kTilePartial = 1, kTileFull = 2, kTileCausal = 3 };

constexpr int kTileThreads = 512, kTileWaves = kTileThreads / 64;
constexpr int kMaxOwn = 1024;         // own tile length
constexpr int64_t kMaxRowTiles = 16384;  // tiles of a row whose classes fit in LDS
constexpr int kFewRuns = 2;  // up to here the compares cost no more than the sieve

struct OwnRuns {
  int64_t doc[kMaxOwn];
  int bound[kMaxOwn];
  uint32_t ids[2048];  // 65536 bits by hash of the id: 128 runs leave 0.2% of others a hit
  int n;

  __device__ static __forceinline__ uint32_t hash(int64_t d) {
    return (uint32_t)(((uint64_t)d * 0x9E3779B97F4A7C15ull) >> 48);
  }
  __device__ __forceinline__ bool may_hold(int64_t d) const {
    const uint32_t h = hash(d);
    return (ids[h >> 5] >> (h & 31)) & 1;
  }
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
  for (int i = tid; i < 2048; i += kTileThreads) runs.ids[i] = 0;
  __syncthreads();
  for (int64_t p = own0 + tid; p < own_end; p += kTileThreads) {
    const int64_t d = doc[p];
    const bool edge = by_kv ? p == own0 || doc[p - 1] != d : p + 1 == own_end || doc[p + 1] != d;
    // One atomic a wave for its runs' places.
    const uint64_t edges = __builtin_amdgcn_ballot_w64(edge);
    int at = 0;
    if (edges != 0 && lane == __builtin_ctzll(edges))
      at = atomicAdd(&runs.n, __builtin_popcountll(edges));
    at = __shfl(at, edges != 0 ? __builtin_ctzll(edges) : 0);
    if (edge) {
      const int i = at + __builtin_popcountll(edges & ((1ull << lane) - 1ull));
      runs.doc[i] = d;
      runs.bound[i] = (int)p;
      const uint32_t h = OwnRuns::hash(d);
      atomicOr(&runs.ids[h >> 5], 1u << (h & 31));
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
    bool visit = !never;
    if (visit && n > kFewRuns) {
      bool hit = false;
      for (int j = lane; j < other; j += 64) {
        const int64_t p = p0 + j;
        if (p < s) hit |= runs.may_hold(j < 64 ? first : doc[p]);
      }
      visit = __builtin_amdgcn_ballot_w64(hit) != 0;
    }
    if (visit) {
      bool any = false, all = whole, one = true;
      bool decided = false;  // (of more than one run: never full)
      for (int j0 = 0; j0 < other && !decided; j0 += 64) {
        const int j = j0 + lane;
        const int64_t p = p0 + j;
        const bool mine = j < other, in = mine && p < s;
        const int64_t d = j < 64 ? first : in ? doc[p] : 0;
        auto compare = [&](int r) {
          const bool side = in && (by_kv ? p >= runs.bound[r] : p <= runs.bound[r]);
          const bool same = d == runs.doc[r];
          any |= side & same;
          one &= !side | same;
        };
        for (int r0 = 0; r0 < n && !decided; r0 += 16) {
          const int r1 = min(r0 + 16, n);
          int r = r0;
          for (; r + 8 <= r1; r += 8) {  // (eight runs read at a time)
#pragma unroll
            for (int i = 0; i < 8; ++i) compare(r + i);
          }
          for (; r < r1; ++r) compare(r);
          decided = n > 1 && __builtin_amdgcn_ballot_w64(any) != 0 &&
                    (!causal_class || __builtin_amdgcn_ballot_w64(!one) != 0);
        }
        all &= !mine || (in && d == runs.doc[0] && (by_kv ? p >= far : p <= far));
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
