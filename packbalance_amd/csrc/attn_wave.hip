// Document-masked GQA attention on small grids, head dims to 64 (multiples of
// 8), any sequence length, for gfx950: waves that never wait for each other.
//
// A pack of a few documents gives lists of one to a few dozen 32 x 32 tiles,
// and at head dim 64 a tile is 8 to 16 MFMAs, so in the workgroup kernels
// (attn_fwd_pipe and the backward's) the barrier of every 32-row step, the
// rows and columns of a 128 x 64 plan tile that hold no allowed pair, and the
// workgroup with the longest list set the time, not the matrix cores:
// [4, 2048], 12 / 4 heads: dK/dV 107 us for 108 steps of the longest list
// where the mean is 36.
//
// Here a workgroup of one to eight waves owns ONE 32-row tile (of queries, or of
// KV rows for dK/dV).  Plans are 32 x 32, so only tiles that hold a pair are
// visited.  The list is shared out evenly over the waves (wave_share), each
// wave streams its own share with its own LDS ring (DMA one step ahead, waited
// for with vmcnt alone) and no barrier, and the waves' results meet once, in
// the ring's LDS, at the end -- so long lists need no fp32 partials in HBM and
// no merge kernel.  Waves without a share leave at once.  Latency is covered
// by the other waves of the SIMD (three in the forward and dQ, two in dK/dV),
// not by software pipelining.  K, V (or Q, dO) tiles are read once per wave
// from L2 instead of once per workgroup, which is why larger grids and longer
// sequences keep the workgroup kernels (wave_tiles).
//
// Measured in captured launches, workgroup -> wave kernels with their merges, 12 / 4
// heads, D 64: [4, 2048] forward 41 -> 27 us, backward 135 -> 71 us; [2, 2048] 25 ->
// 16 and 59 -> 43 us.  What is left is latency: there the VALU is active 19 to 23%
// of the waves' time and the matrix cores 8 to 9% of the kernels'.
//
// MFMA layouts, masks and log2-domain lse as in attn_fwd.hip / attn_bwd.hip.
#include "attn_args.hpp"

namespace pb {
namespace attn {
namespace {

// Waves per workgroup of the forward and dQ, and the least steps worth another
// wave.  Two were the fastest or within 3% of it from 768 to 12288 tiles, short
// and long lists ([4, 2048], 12 heads: forward 30 / 27 / 34 us and dQ 35 / 33 /
// 42 us with 1 / 2 / 4 waves): more leave most of a workgroup's LDS to waves
// without a share.  Up to kFewQ tiles (three per CU) the CUs have room, the
// longest list sets the time, and four are faster: forward of [1, 2048], 4
// heads, one document 21.2 -> 13.4 us (the workgroup kernels 18.7), [1, 2048],
// 12 heads 22.5 -> 17.1 (30.3); at 1152 tiles ([1, 3072], 12 heads, documents of
// about 100) 14.1 -> 15.3.
constexpr int kFewQ = 768;
constexpr int kWaveLeast = 6, kFewLeast = 4;  // kFewLeast: four waves of the forward and dQ
constexpr int kTB = 32 * 64 * 2;   // bytes of one 32 x 64 bf16 tile
constexpr int NDK = 4, NDB = 2;    // 16-wide k steps and 32-wide blocks of the head dim
using Dma = TileDma<64, 32, 64>;   // one wave copies a tile: four 1 KiB instructions

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Wave w's part [i0, i1) of n steps: at most NW waves of at least LEAST steps
// (all but the first wave cost a prologue and a merge).  pb_attn_plan leaves no
// list empty, but a caller's plan may: the first wave then has no step.
// Returns the number of waves that have a share.
template <int NW, int LEAST = kWaveLeast>
__device__ __forceinline__ int wave_share(int n, int w, int &i0, int &i1) {
  const int nw = max(1, min(NW, n / LEAST));
  i0 = n * w / nw;
  i1 = n * (w + 1) / nw;
  return nw;
}

// Row fragments of a row this lane owns for the whole kernel.
__device__ __forceinline__ void own_frags(const bf16_t *row, int hh, int d, bf16x8_t (&f)[NDK]) {
#pragma unroll
  for (int dk = 0; dk < NDK; ++dk) {
    const int c = 16 * dk + 8 * hh;
    if (c < d) f[dk] = *reinterpret_cast<const bf16x8_t *>(row + c);
    else f[dk] = bf16x8_t{};
  }
}

// LDS offsets of a swizzled 32 x 64 tile: row fragments (as own_frags) and the
// two transposing reads of a column fragment (see lds_col_frag).
struct FragOffs {
  int row[NDK], col[NDB][2];
  __device__ __forceinline__ void init(int lane) {
    const int j = lane & 15, g = lane >> 4, h = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int dk = 0; dk < NDK; ++dk) row[dk] = SwzTile<64>::off(l32, 16 * dk + 8 * h);
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const int c = 32 * db + 16 * (g & 1) + 4 * (j & 3), r = 4 * h + (j >> 2);
      col[db][0] = SwzTile<64>::off(r, c);
      col[db][1] = SwzTile<64>::off(r + 8, c);
    }
  }
  __device__ __forceinline__ bf16x8_t rfrag(const char *t, int dk) const {
    return *reinterpret_cast<const bf16x8_t *>(t + row[dk]);
  }
  // Column fragment of head-dim block db at tile rows 16 kk + pi(h, s).
  __device__ __forceinline__ bf16x8_t cfrag(const char *t, int kk, int db) const {
    const char *base = t + kk * 16 * 64 * 2;
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(base + col[db][0]));
    const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t *)(base + col[db][1]));
    typedef short i16x8_t __attribute__((ext_vector_type(8)));
    i16x8_t r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return *reinterpret_cast<bf16x8_t *>(&r);
  }
};

// Element mask of a tile that is not FULL.  `own` is the lane's row position
// (a query when QMAJOR, a KV row otherwise), `r0` the first row of the other
// axis, `od` the lane's document, `docs` the other axis' 32 documents in LDS.
// `diag`: the tile may hold pairs with kv > q.
template <bool QMAJOR>
__device__ __forceinline__ void mask_tile(f32x16_t &s, bool causal, bool diag, int own, int r0,
                                          int hh, int64_t od, const int64_t *docs) {
  const int rel = own - r0 - 4 * hh;  // own position in the rows 8(j/4) + j%4
  if (!causal) {
    int64_t d[16];
    lds_docs16(docs, hh, d);
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = d[j] == od ? s[j] : -INFINITY;
  }
  if (diag) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int c = 8 * (j >> 2) + (j & 3);
      s[j] = (QMAJOR ? c <= rel : rel <= c) ? s[j] : -INFINITY;
    }
  }
}

// A lane's accumulators to and from its wave's LDS (16-byte vectors, lane
// innermost: conflict-free), 4 KiB per 16 registers.
__device__ __forceinline__ void put16(char *dst, int lane, const f32x16_t &v) {
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<f32x4_t *>(dst + (g * 64 + lane) * 16) =
        f32x4_t{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
}
__device__ __forceinline__ void add16(const char *src, int lane, float f, f32x16_t &v) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4_t x = *reinterpret_cast<const f32x4_t *>(src + (g * 64 + lane) * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[4 * g + i] += f * x[i];
  }
}

// A query row's 64 output columns (lane <-> query, register j of block db <->
// column 32 db + 8(j/4) + 4 hh + j%4), scaled and rounded once.
__device__ __forceinline__ void store_row(bf16_t *row, int hh, int d, const f32x16_t (&v)[NDB],
                                          float f) {
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      if (32 * db + 8 * jq >= d) continue;
      bf16x4_t o4;
#pragma unroll
      for (int x = 0; x < 4; ++x) o4[x] = (bf16_t)(v[db][4 * jq + x] * f);
      *reinterpret_cast<bf16x4_t *>(row + 32 * db + 8 * jq + 4 * hh) = o4;
    }
}

__device__ __forceinline__ void pack2(bf16x8_t (&f)[2], int j, float x0, float x1) {
  f[j >> 3][j & 7] = (bf16_t)x0;
  f[j >> 3][(j & 7) + 1] = (bf16_t)x1;
}

// All but the newest N vector-memory operations of this wave have landed; no
// instruction moves across.
template <int N>
__device__ __forceinline__ void settle() {
  __builtin_amdgcn_sched_barrier(0);
  wait_vmcnt<N>();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// ---------------------------------------------------------------- forward
// Per step: S^T = K Q^T, online softmax with the running max moved when it
// grows by more than FwdArgs::tau (log2 units), O^T += V^T P^T.  The next step's K goes
// to the one K slot as soon as S has read it, its V to the other of two V
// slots: 12 KiB a wave, three waves per SIMD.  (K fragments loaded straight
// into registers, 32 rows of 16 bytes an instruction, measured 2x slower.)
template <int NW, int LEAST>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3, 3)))
void attn_fwd_wave(FwdArgs a) {
  __shared__ __align__(16) char ks[NW][kTB], vs0[NW][kTB], vs1[NW][kTB];
  __shared__ __align__(16) int64_t kd0[NW][32], kd1[NW][32];
  __shared__ float ml[NW][2][64];
  const int lane = threadIdx.x & 63, hh = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int qt, b, h;
  decode_q_major((int)blockIdx.x, a.nqt, a.B, a.Hq, a.Hkv, qt, b, h);
  const int n = a.cnt[b * a.nqt + qt];
  int i0, i1;
  const int nw = wave_share<NW, LEAST>(n, wave, i0, i1);
  if (wave >= nw) return;
  const int m = i1 - i0;  // at most 64: n <= kWaveMaxS / 32 over two waves
  const int S = a.S, hk = h / (a.Hq / a.Hkv);
  const float sl2 = a.sl2;
  const int32_t *lst = a.list + ((int64_t)b * a.nqt + qt) * a.nkt + i0;
  const int ev = lst[max(min(lane, m - 1), 0)];
  auto entry = [&](int i) { return __builtin_amdgcn_readlane(ev, min(i, m - 1)); };
  const auto krs = buf_rsrc(a.k + b * a.k_sb + hk * a.k_sh, 0x7fffffff);
  const auto vrs = buf_rsrc(a.v + b * a.v_sb + hk * a.v_sh, 0x7fffffff);
  const auto drs = buf_rsrc(a.doc + b * a.doc_sb, 0x7fffffff);
  const uint32_t kss2 = (uint32_t)(a.k_ss * 2), vss2 = (uint32_t)(a.v_ss * 2);
  uint32_t koff[Dma::NDMA], voff[Dma::NDMA];
  const int drow = Dma::offsets_gen(a.k_ss, 0, lane, a.D, koff);
  Dma::offsets_gen(a.v_ss, 0, lane, a.D, voff);
  FragOffs fo;
  fo.init(lane);

  const int qi = qt * 32 + l32;
  const bool qv = qi < S;
  const int qr = qv ? qi : S - 1;
  bf16x8_t qf[NDK];
  own_frags(a.q + b * a.q_sb + h * a.q_sh + (int64_t)qr * a.q_ss, hh, a.D, qf);
  const int64_t qdoc = a.doc[b * a.doc_sb + qr];

  f32x16_t oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) oacc[db] = zero16();
  float m_run = -INFINITY, m_use = 0.f, l_run = 0.f;

  char *const kt = ks[wave], *const v0 = vs0[wave], *const v1 = vs1[wave];
  // One step's DMA: documents and K (5 operations), then V (4).
  auto fetch = [&](int i, char *vdst, int64_t *ddst) {
    const int r0 = plan_tile(entry(i)) * 32;
    dma_docs_gen(drs, r0, S, lane, ddst);
    Dma::copy_gen(krs, (uint32_t)r0 * kss2, koff, drow, S - r0, kt, 0);
    Dma::copy_gen(vrs, (uint32_t)r0 * vss2, voff, drow, S - r0, vdst, 0);
  };
  // Step i from V slot vt and documents kd; fetches step i + 1 (past the last
  // step the last one again, which nobody reads) into vn and dn.
  auto step = [&](int i, const char *vt, const int64_t *kd, char *vn, int64_t *dn) {
    const int e = entry(i), t = plan_tile(e);
    settle<4>();  // this step's documents and K
    f32x16_t s = zero16();
#pragma unroll
    for (int dk = 0; dk < NDK; ++dk) s = mfma32(fo.rfrag(kt, dk), qf[dk], s);
    __builtin_amdgcn_sched_barrier(0);  // K is read: its slot takes the next step's
    fetch(i + 1, vn, dn);
    if (!plan_full(e)) mask_tile<true>(s, plan_causal(e), t == qt, qi, t * 32, hh, qdoc, kd);
    float m0 = s[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) m0 = fmaxf(m0, s[j]);
    const float m1 = xor32_max(m0) * sl2;
    const bool move = m1 > m_run + a.tau;
    if (__builtin_amdgcn_ballot_w64(move) != 0) {
      const float mn = move ? m1 : m_run;
      const float alpha = mn == m_run ? 1.f : fast_exp2(m_run - mn);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) oacc[db] *= alpha;
      m_run = mn;
      m_use = mn == -INFINITY ? 0.f : mn;
    }
    bf16x8_t pf[2];
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
      const float p0 = fast_exp2(fmaf(s[j], sl2, -m_use));
      const float p1 = fast_exp2(fmaf(s[j + 1], sl2, -m_use));
      l0 += p0;
      l1 += p1;
      pack2(pf, j, p0, p1);
    }
    l_run += l0 + l1;
    settle<9>();  // this step's V
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < NDB; ++db) oacc[db] = mfma32(fo.cfrag(vt, kk, db), pf[kk], oacc[db]);
  };
  if (m > 0) fetch(0, v0, kd0[wave]);
  int i = 0;
  for (; i + 2 <= m; i += 2) {
    step(i, v0, kd0[wave], v1, kd1[wave]);
    step(i + 1, v1, kd1[wave], v0, kd0[wave]);
  }
  if (i < m) step(i, v0, kd0[wave], v1, kd1[wave]);
  settle<0>();  // the fetch past the last step, before its LDS is used again or given back
  if (nw > 1) {
    if (wave > 0) {
      put16(v0, lane, oacc[0]);
      put16(v1, lane, oacc[1]);
      ml[wave][0][lane] = m_run;
      ml[wave][1][lane] = l_run;
    }
    __syncthreads();
    if (wave > 0) return;
    float mx = m_run;
    for (int w = 1; w < nw; ++w) mx = fmaxf(mx, ml[w][0][lane]);
    const float mu = mx == -INFINITY ? 0.f : mx;
    const float f0 = fast_exp2(m_run - mu);
    l_run *= f0;
#pragma unroll
    for (int db = 0; db < NDB; ++db) oacc[db] *= f0;
    for (int w = 1; w < nw; ++w) {
      const float f = fast_exp2(ml[w][0][lane] - mu);
      l_run += f * ml[w][1][lane];
      add16(vs0[w], lane, f, oacc[0]);
      add16(vs1[w], lane, f, oacc[1]);
    }
    m_run = mx;
  }
  const float lt = xor32_sum(l_run);
  if (!qv) return;
  store_row(a.o + b * a.o_sb + (int64_t)qi * a.o_ss + h * a.o_sh, hh, a.D, oacc,
            lt > 0.f ? 1.0f / lt : 0.f);
  if (hh == 0)
    a.lse[((int64_t)b * a.Hq + h) * S + qi] = lt > 0.f ? m_run + fast_log2(lt) : -INFINITY;
}

// ---------------------------------------------------------------- dQ (+ delta)
// Per step: S^T = K Q^T and dP^T = V dO^T, dS^T = P (dP - delta), dQ^T += K^T
// dS^T with K^T read from the same K tile.  The next step's V goes to the one
// V slot as soon as dP has read it, its K to the other of two K slots.
template <int NW, int LEAST>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3, 3)))
void attn_bwd_dq_wave(BwdArgs a) {
  __shared__ __align__(16) char ks0[NW][kTB], ks1[NW][kTB], vs[NW][kTB];
  __shared__ __align__(16) int64_t kd0[NW][32], kd1[NW][32];
  const int lane = threadIdx.x & 63, hh = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int qt, b, h;
  decode_q_major((int)blockIdx.x, a.nqt_dq, a.B, a.Hq, a.Hkv, qt, b, h);
  const int n = a.qcnt[b * a.nqt_dq + qt];
  int i0, i1;
  const int nw = wave_share<NW, LEAST>(n, wave, i0, i1);
  if (wave >= nw) return;
  const int m = i1 - i0;
  const int S = a.S, hk = h / (a.Hq / a.Hkv);
  const float sl2 = a.sl2;
  const int32_t *lst = a.qlist + ((int64_t)b * a.nqt_dq + qt) * a.nkt_dq + i0;
  const int ev = lst[max(min(lane, m - 1), 0)];
  auto entry = [&](int i) { return __builtin_amdgcn_readlane(ev, min(i, m - 1)); };
  const auto krs = buf_rsrc(a.k.row(b, hk, 0), 0x7fffffff);
  const auto vrs = buf_rsrc(a.v.row(b, hk, 0), 0x7fffffff);
  const auto drs = buf_rsrc(a.doc + b * a.doc_sb, 0x7fffffff);
  const uint32_t kss2 = (uint32_t)(a.k.ss * 2), vss2 = (uint32_t)(a.v.ss * 2);
  uint32_t koff[Dma::NDMA], voff[Dma::NDMA];
  const int drow = Dma::offsets_gen(a.k.ss, 0, lane, a.D, koff);
  Dma::offsets_gen(a.v.ss, 0, lane, a.D, voff);
  FragOffs fo;
  fo.init(lane);

  const int qi = qt * 32 + l32;
  const bool qv = qi < S;
  const int qr = qv ? qi : S - 1;
  const int64_t row_o = ((int64_t)b * a.Hq + h) * S + qr;
  const int64_t qdoc = a.doc[b * a.doc_sb + qr];
  const float lse = a.lse[row_o];
  bf16x8_t qf[NDK], gf[NDK];
  own_frags(a.q.row(b, h, qr), hh, a.D, qf);
  own_frags(a.dout.row(b, h, qr), hh, a.D, gf);
  float dlt = 0.f;
  {
    bf16x8_t of[NDK];
    own_frags(a.o.row(b, h, qr), hh, a.D, of);
#pragma unroll
    for (int dk = 0; dk < NDK; ++dk)
#pragma unroll
      for (int i = 0; i < 8; ++i) dlt += (float)gf[dk][i] * (float)of[dk][i];
    dlt = xor32_sum(dlt);  // the lane halves hold complementary slices of the row
    if (wave == 0 && qv && hh == 0) a.delta[row_o] = dlt;
  }
  f32x16_t acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();

  char *const k0 = ks0[wave], *const k1 = ks1[wave], *const vt = vs[wave];
  auto fetch = [&](int i, char *kdst, int64_t *ddst) {
    const int r0 = plan_tile(entry(i)) * 32;
    dma_docs_gen(drs, r0, S, lane, ddst);
    Dma::copy_gen(krs, (uint32_t)r0 * kss2, koff, drow, S - r0, kdst, 0);
    Dma::copy_gen(vrs, (uint32_t)r0 * vss2, voff, drow, S - r0, vt, 0);
  };
  auto step = [&](int i, const char *kt, const int64_t *kd, char *kn, int64_t *dn) {
    const int e = entry(i), t = plan_tile(e);
    settle<0>();  // this step's documents, K and V
    f32x16_t s = zero16(), p = zero16();
#pragma unroll
    for (int dk = 0; dk < NDK; ++dk) {
      s = mfma32(fo.rfrag(kt, dk), qf[dk], s);
      p = mfma32(fo.rfrag(vt, dk), gf[dk], p);
    }
    __builtin_amdgcn_sched_barrier(0);  // V is read: its slot takes the next step's
    fetch(i + 1, kn, dn);
    if (!plan_full(e)) mask_tile<true>(s, plan_causal(e), t == qt, qi, t * 32, hh, qdoc, kd);
    bf16x8_t ds[2];
#pragma unroll
    for (int j = 0; j < 16; j += 2)
      pack2(ds, j, fast_exp2(fmaf(s[j], sl2, -lse)) * (p[j] - dlt),
            fast_exp2(fmaf(s[j + 1], sl2, -lse)) * (p[j + 1] - dlt));
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] = mfma32(fo.cfrag(kt, kk, db), ds[kk], acc[db]);
  };
  if (m > 0) fetch(0, k0, kd0[wave]);
  int i = 0;
  for (; i + 2 <= m; i += 2) {
    step(i, k0, kd0[wave], k1, kd1[wave]);
    step(i + 1, k1, kd1[wave], k0, kd0[wave]);
  }
  if (i < m) step(i, k0, kd0[wave], k1, kd1[wave]);
  settle<0>();
  if (nw > 1) {
    if (wave > 0) {
      put16(k0, lane, acc[0]);
      put16(k1, lane, acc[1]);
    }
    __syncthreads();
    if (wave > 0) return;
    for (int w = 1; w < nw; ++w) {
      add16(ks0[w], lane, 1.f, acc[0]);
      add16(ks1[w], lane, 1.f, acc[1]);
    }
  }
  if (qv) store_row(a.dq.row(b, h, qi), hh, a.D, acc, a.scale);
}

// ---------------------------------------------------------------- dK, dV
// Lane <-> KV row.  The steps are (query tile of the list, query head of the
// GQA group), heads inner; per step S = Q K^T, dP = dO V^T, dV += P^T dO and
// dK += dS^T Q from one Q and one dO tile (two-slot rings, DMA a step ahead).
// Query rows past the end arrive as zero Q, dO, lse and delta and add nothing.
template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_bwd_dkdv_wave(BwdArgs a) {
  __shared__ __align__(16) char qs0[NW][kTB], qs1[NW][kTB], gs0[NW][kTB], gs1[NW][kTB];
  __shared__ __align__(16) float ld0[NW][64], ld1[NW][64];  // lse[32], delta[32]
  __shared__ __align__(16) int64_t qd0[NW][32], qd1[NW][32];
  const int lane = threadIdx.x & 63, hh = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.Hq / a.Hkv;
  // Early KV tiles (the longest lists) of every (pack, KV head) first, each
  // pair on one XCD, whose L2 then holds its Q and dO rows.
  const int npairs = a.B * a.Hkv;
  int kt, pair;
  if (npairs % 8 == 0) {
    const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3, np8 = npairs >> 3;
    kt = j / np8;
    pair = (j - kt * np8) * 8 + x;
  } else {
    kt = (int)blockIdx.x / npairs;
    pair = (int)blockIdx.x - kt * npairs;
  }
  const int b = pair / a.Hkv, hk = pair - b * a.Hkv;
  const int cnt = a.kcnt[b * a.nkt_kv + kt];
  int t0, t1;
  const int nw = wave_share<NW>(cnt * G, wave, t0, t1);
  if (wave >= nw) return;
  const int S = a.S;
  const float sl2 = a.sl2;
  // This wave's query tiles: list entries u0 .. (at most 128 of them).
  const int u0 = t0 / G;
  const int32_t *lst = a.klist + ((int64_t)b * a.nkt_kv + kt) * a.nqt_kv;
  const int ev0 = lst[max(min(u0 + lane, cnt - 1), 0)];
  const int ev1 = lst[max(min(u0 + 64 + lane, cnt - 1), 0)];
  auto entry = [&](int i) { return __builtin_amdgcn_readlane(i < 64 ? ev0 : ev1, i & 63); };
  const int h0 = hk * G;
  const auto qrs = buf_rsrc(a.q.row(b, h0, 0), 0x7fffffff);
  const auto grs = buf_rsrc(a.dout.row(b, h0, 0), 0x7fffffff);
  const auto lrs = buf_rsrc(a.lse + ((int64_t)b * a.Hq + h0) * S, 0x7fffffff);
  const auto trs = buf_rsrc(a.delta + ((int64_t)b * a.Hq + h0) * S, 0x7fffffff);
  const auto drs = buf_rsrc(a.doc + b * a.doc_sb, 0x7fffffff);
  const uint32_t qsh2 = (uint32_t)(a.q.sh * 2), qss2 = (uint32_t)(a.q.ss * 2);
  const uint32_t gsh2 = (uint32_t)(a.dout.sh * 2), gss2 = (uint32_t)(a.dout.ss * 2);
  uint32_t qoff[Dma::NDMA], goff[Dma::NDMA];
  const int drow = Dma::offsets_gen(a.q.ss, 0, lane, a.D, qoff);
  Dma::offsets_gen(a.dout.ss, 0, lane, a.D, goff);
  FragOffs fo;
  fo.init(lane);

  const int kv = kt * 32 + l32;
  const bool kvv = kv < S;
  const int kvr = kvv ? kv : S - 1;
  const int64_t kvdoc = a.doc[b * a.doc_sb + kvr];
  bf16x8_t kf[NDK], vf[NDK];
  own_frags(a.k.row(b, hk, kvr), hh, a.D, kf);
  own_frags(a.v.row(b, hk, kvr), hh, a.D, vf);
  f32x16_t dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) dk[db] = dv[db] = zero16();

  // The step to fetch next: (list entry u, head g); past the share's end the
  // last one is fetched again, into a slot nobody reads.
  int fu = 0, fg = t0 - u0 * G, ft = t0;
  auto fetch = [&](char *qd, char *gd, float *ld, int64_t *dd) {
    const int r0 = plan_tile(entry(fu)) * 32, left = S - r0;
    const uint32_t ro = ((uint32_t)fg * (uint32_t)S + (uint32_t)r0) * 4u;
    const uint32_t rv = l32 < left ? 4u * l32 : kDmaZero;
    if (lane < 32) dma4_rs(lrs, ro, rv, ld);   // lane i writes LDS float i
    if (lane >= 32) dma4_rs(trs, ro, rv, ld);
    dma_docs_gen(drs, r0, S, lane, dd);
    Dma::copy_gen(qrs, (uint32_t)fg * qsh2 + (uint32_t)r0 * qss2, qoff, drow, left, qd, 0);
    Dma::copy_gen(grs, (uint32_t)fg * gsh2 + (uint32_t)r0 * gss2, goff, drow, left, gd, 0);
    if (ft + 1 < t1) {
      ++ft;
      if (++fg == G) {
        fg = 0;
        ++fu;
      }
    }
  };
  int cu = 0, cg = t0 - u0 * G;  // the step being computed
  auto step = [&](const char *qt_, const char *gt, const float *ld, const int64_t *qd) {
    const int e = entry(cu), t = plan_tile(e);
    if (++cg == G) {
      cg = 0;
      ++cu;
    }
    f32x16_t s = zero16(), p = zero16();
#pragma unroll
    for (int d = 0; d < NDK; ++d) s = mfma32(fo.rfrag(qt_, d), kf[d], s);
#pragma unroll
    for (int d = 0; d < NDK; ++d) p = mfma32(fo.rfrag(gt, d), vf[d], p);
    float lse[16], dlt[16];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4_t l4 = *reinterpret_cast<const f32x4_t *>(ld + 8 * g + 4 * hh);
      const f32x4_t d4 = *reinterpret_cast<const f32x4_t *>(ld + 32 + 8 * g + 4 * hh);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        lse[4 * g + x] = l4[x];
        dlt[4 * g + x] = d4[x];
      }
    }
    if (!plan_full(e)) mask_tile<false>(s, plan_causal(e), t == kt, kv, t * 32, hh, kvdoc, qd);
    bf16x8_t pf[2], ds[2];
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
      const float p0 = fast_exp2(fmaf(s[j], sl2, -lse[j]));
      const float p1 = fast_exp2(fmaf(s[j + 1], sl2, -lse[j + 1]));
      pack2(pf, j, p0, p1);
      pack2(ds, j, p0 * (p[j] - dlt[j]), p1 * (p[j + 1] - dlt[j + 1]));
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        dv[db] = mfma32(pf[kk], fo.cfrag(gt, kk, db), dv[db]);
        dk[db] = mfma32(ds[kk], fo.cfrag(qt_, kk, db), dk[db]);
      }
  };
  char *q0 = qs0[wave], *q1 = qs1[wave], *g0 = gs0[wave], *g1 = gs1[wave];
  const int m = t1 - t0;
  if (m > 0) fetch(q0, g0, ld0[wave], qd0[wave]);
  int i = 0;
  for (; i + 2 <= m; i += 2) {
    fetch(q1, g1, ld1[wave], qd1[wave]);
    settle<11>();
    step(q0, g0, ld0[wave], qd0[wave]);
    __builtin_amdgcn_sched_barrier(0);
    fetch(q0, g0, ld0[wave], qd0[wave]);
    settle<11>();
    step(q1, g1, ld1[wave], qd1[wave]);
    __builtin_amdgcn_sched_barrier(0);
  }
  settle<0>();
  if (i < m) step(q0, g0, ld0[wave], qd0[wave]);
  // Wave 0 sums and writes dV, wave 1 (wave 0 when alone) dK.
  if (NW > 1 && nw > 1) {
    if (wave != 0) {
      put16(q0, lane, dv[0]);
      put16(q1, lane, dv[1]);
    }
    if (wave != 1) {
      put16(g0, lane, dk[0]);
      put16(g1, lane, dk[1]);
    }
    __syncthreads();
    if (wave > 1) return;
    for (int w = 0; w < nw; ++w) {
      if (wave == 0 && w != 0) {
        add16(qs0[w], lane, 1.f, dv[0]);
        add16(qs1[w], lane, 1.f, dv[1]);
      }
      if (wave == 1 && w != 1) {
        add16(gs0[w], lane, 1.f, dk[0]);
        add16(gs1[w], lane, 1.f, dk[1]);
      }
    }
  }
  // Accumulators: lane <-> head-dim column, register j <-> KV row.
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    const int d = 32 * db + l32;
    if (d >= a.D) continue;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int r = kt * 32 + 8 * (j >> 2) + 4 * hh + (j & 3);
      if (r >= S) continue;
      if (wave == 0) a.dv.row(b, hk, r)[d] = (bf16_t)dv[db][j];
      if (wave == 1 || nw == 1) a.dk.row(b, hk, r)[d] = (bf16_t)(dk[db][j] * a.scale);
    }
  }
}

// A thread moves eight elements of a row.
template <bool TO_DENSE>
__global__ __launch_bounds__(256) void copy_rows(RowCopies a) {
  const RowCopies::Item &c = a.c[blockIdx.y];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int chunks = a.D / 8;
  int64_t r = i / chunks;
  const int x = (int)(i - r * chunks) * 8;
  if (r >= (int64_t)a.B * c.heads * a.S) return;
  const int s = (int)(r % a.S);
  r /= a.S;
  const int h = (int)(r % c.heads), b = (int)(r / c.heads);
  bf16_t *p = c.view + b * c.sb + h * c.sh + s * c.ss + x;
  bf16x8_t *d = reinterpret_cast<bf16x8_t *>(c.dense + 8 * i);
  bf16x8_t v;
  if constexpr (TO_DENSE) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = p[j];
    *d = v;
  } else {
    v = *d;
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = v[j];
  }
}

}  // namespace

int launch_row_copies(const RowCopies &c, bool to_dense, hipStream_t st) {
  int heads = 0;
  for (int i = 0; i < c.n; ++i) heads = c.c[i].heads > heads ? c.c[i].heads : heads;
  const int64_t n = (int64_t)c.B * heads * c.S * (c.D / 8);
  const dim3 g((unsigned)((n + 255) / 256), (unsigned)c.n);
  if (to_dense) hipLaunchKernelGGL(copy_rows<true>, g, dim3(256), 0, st, c);
  else hipLaunchKernelGGL(copy_rows<false>, g, dim3(256), 0, st, c);
  return launch_status("pb_attn(row copies)");
}

// Rows too short for a second wave's part have one wave a query tile (forward of
// one document, 16 / 2 heads: [32, 128] 13.7 -> 10.7 us, [16, 200] 13.6 -> 10.6).
int launch_fwd_wave(const FwdArgs &a, hipStream_t st) {
  const int tiles = a.nqt * a.B * a.Hq;
  const dim3 g((unsigned)tiles);
  if (tiles <= kFewQ && a.nkt >= 2 * kFewLeast)
    hipLaunchKernelGGL((attn_fwd_wave<4, kFewLeast>), g, dim3(256), 0, st, a);
  else if (a.nkt >= 2 * kWaveLeast)
    hipLaunchKernelGGL((attn_fwd_wave<2, kWaveLeast>), g, dim3(128), 0, st, a);
  else
    hipLaunchKernelGGL((attn_fwd_wave<1, kWaveLeast>), g, dim3(64), 0, st, a);
  return launch_status("pb_attn_fwd");
}

int launch_bwd_wave(const BwdArgs &a, hipStream_t st) {
  // dQ first: it also writes delta = rowsum(dO * O), which dK/dV reads.
  const int qtiles = a.nqt_dq * a.B * a.Hq;
  const dim3 gq((unsigned)qtiles);
  if (qtiles <= kFewQ && a.nkt_dq >= 2 * kFewLeast)
    hipLaunchKernelGGL((attn_bwd_dq_wave<4, kFewLeast>), gq, dim3(256), 0, st, a);
  else if (a.nkt_dq >= 2 * kWaveLeast)
    hipLaunchKernelGGL((attn_bwd_dq_wave<2, kWaveLeast>), gq, dim3(128), 0, st, a);
  else
    hipLaunchKernelGGL((attn_bwd_dq_wave<1, kWaveLeast>), gq, dim3(64), 0, st, a);
  const int rc = launch_status("pb_attn_bwd(dq)");
  if (rc) return rc;
  // Waves per workgroup by the number of KV tiles: at 1024 tiles (2048 waves
  // are resident) the longest list still sets the time and four waves are
  // fastest ([2, 2048], 12 / 4 heads: 71 / 41 / 27 us with 1 / 2 / 4 waves;
  // [4, 2048]: 63 / 39 / 37 us), at 4096 two ([16, 2048]: 151 / 140 / 165 us),
  // beyond that one ([8, 2048], 16 / 16 heads: 87 / 120 / 185 us).  Up to one
  // workgroup per CU eight, and to 384 tiles with long lists: one document, dQ and
  // dK/dV with 4 / 8: [1, 2048], 9 / 3 heads 65 / 53 us (workgroup kernels 67);
  // 384 tiles: [1, 3072], 16 / 4 132 / 109 (125), but [1, 2048], 6 / 6 38 / 45.
  // No more waves than the longest list has parts of kWaveLeast steps (up to one
  // workgroup per CU, where idle waves cost less, no twice as many).  Backward of
  // one document, 12 / 4 heads, with these counts in dQ and dK/dV, before / after:
  // [64, 128] (KV tiles of up to 12 steps) 43.8 / 35.5 us, [32, 200] 45.2 / 35.1,
  // [1, 64] 15.5 / 14.5; [16, 384], 4 / 4 heads 28.9 / 26.1.
  const int64_t tiles = (int64_t)a.nkt_kv * a.B * a.Hkv;
  const dim3 gk((unsigned)tiles);
  const int longest = a.nqt_kv * (a.Hq / a.Hkv);  // steps
  int nw = tiles <= 256 || (tiles <= 384 && longest >= 288) ? 8
           : tiles <= 1024                                  ? 4
           : tiles <= 4096                                  ? 2
                                                            : 1;
  const int parts = longest / kWaveLeast;
  while (nw > 1 && (tiles <= 256 ? nw / 2 >= parts : nw > parts)) nw /= 2;
  if (nw == 8) hipLaunchKernelGGL(attn_bwd_dkdv_wave<8>, gk, dim3(512), 0, st, a);
  else if (nw == 4) hipLaunchKernelGGL(attn_bwd_dkdv_wave<4>, gk, dim3(256), 0, st, a);
  else if (nw == 2) hipLaunchKernelGGL(attn_bwd_dkdv_wave<2>, gk, dim3(128), 0, st, a);
  else hipLaunchKernelGGL(attn_bwd_dkdv_wave<1>, gk, dim3(64), 0, st, a);
  return launch_status("pb_attn_bwd(dkdv)");
}

}  // namespace attn
}  // namespace pb
