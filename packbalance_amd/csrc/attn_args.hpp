// Kernel arguments of the bf16 attention kernels, shared by the workgroup
// kernels (attn_fwd.hip, attn_bwd.hip) and the wave kernels (attn_wave.hip).
#pragma once

#include "attn_common.hpp"

namespace pb {
namespace attn {

struct FwdArgs {
  const bf16_t *q;
  int64_t q_sb, q_sh, q_ss;
  const bf16_t *k;
  int64_t k_sb, k_sh, k_ss;
  const bf16_t *v;
  int64_t v_sb, v_sh, v_ss;
  bf16_t *o;
  int64_t o_sb, o_sh, o_ss;
  float *lse;  // [B][Hq][S], log2 domain of the scaled scores
  const int64_t *doc;
  int64_t doc_sb;
  const int32_t *cnt;   // [B][nqt]
  const int32_t *list;  // [B][nqt][nkt]
  int B, Hq, Hkv, S, D, nqt, nkt;
  float sl2;  // softmax scale * log2(e)
  int vec;    // 16-byte global access allowed
  // Growth of a row's running max (log2 units) that attn_fwd_wave leaves in the
  // exponentials; 0 keeps the max exact (see softmax state in attn_fwd_pipe).
  float tau;
  // KV split (pipelined kernel): chunk = KV tiles per workgroup (0: whole
  // list); bm = query rows per tile; partial outputs [split][B][Hq][S][D]
  // and log-sum-exps [split][B][Hq][S], fp32.
  int chunk, bm;
  float *part_o, *part_lse;
};

struct View {
  bf16_t *p;
  int64_t sb, sh, ss;
  __device__ __forceinline__ bf16_t *row(int b, int h, int64_t s) const {
    return p + b * sb + h * sh + s * ss;
  }
};

struct BwdArgs {
  View q, k, v, o, dout, dq, dk, dv;
  const float *lse;
  float *delta;
  const int64_t *doc;
  int64_t doc_sb;
  const int32_t *qcnt, *qlist;  // dQ plan (by query tile)
  const int32_t *kcnt, *klist;  // dK/dV plan (by KV tile)
  float *dk_part, *dv_part;     // split: fp32 [B][Hq][S][D] partials
  // split, pipelined kernel: a KV tile whose list has at least kv_chunk steps
  // is walked by two workgroups (first and second half of its steps); the
  // second writes its partials here.  0: whole lists, these are unused.
  float *dk_part2, *dv_part2;
  int kv_chunk, kv_tile;
  // dQ KV split: KV tiles per workgroup (0: whole list), unscaled fp32 dQ
  // partials [split][B][Hq][S][D] of query tiles with more than one chunk.
  int dq_chunk;
  float *dq_part;
  // Kept dS blocks (AttnConfig::ds): the region of pack b, KV head hk starts
  // at ds + (b * Hkv + hk) * ds_pair bytes.
  char *ds;
  int64_t ds_pair;
  int B, Hq, Hkv, S, D;
  int nqt_dq, nkt_dq, nqt_kv, nkt_kv;
  float sl2, scale;
  int vec;
};

// Views that the wave kernels cannot take (rows that are not 16-byte aligned, or
// too far apart for the DMA's offsets) are copied to dense [B][H][S][D] rows
// first, outputs back afterwards: on 32 x 32 plans nothing else runs, and the
// register-staged kernels with one wave per 32-row tile took up to twice as long
// as on their own tiles.  Misaligned [4, 2048], 12 / 4 heads, D 64, one document,
// us, register-staged on 64 x 64 tiles / on 32 x 32 / copied: forward 174 / 367 /
// 74, backward 842 / 1350 / 174.
struct RowCopies {
  struct Item {
    bf16_t *view, *dense;
    int64_t sb, sh, ss;
    int heads;
  } c[5];
  int n, B, S, D;
  char *next;  // first free byte of the workspace

  RowCopies(int b, int s, int d, void *ws) : n(0), B(b), S(s), D(d) {
    next = reinterpret_cast<char *>((reinterpret_cast<uintptr_t>(ws) + 15) & ~(uintptr_t)15);
  }
  // Adds a view; returns its dense rows, whose strides it writes to sb, sh, ss.
  bf16_t *add_at(char *at, const pb_bhsd &v, int heads, int64_t &sb, int64_t &sh, int64_t &ss) {
    bf16_t *dense = reinterpret_cast<bf16_t *>(at);
    c[n++] = {static_cast<bf16_t *>(v.data), dense, v.stride_b, v.stride_h, v.stride_s, heads};
    ss = D;
    sh = (int64_t)S * D;
    sb = heads * sh;
    next = at + B * sb * 2;
    return dense;
  }
  bf16_t *add(const pb_bhsd &v, int heads, int64_t &sb, int64_t &sh, int64_t &ss) {
    return add_at(next, v, heads, sb, sh, ss);
  }
};
int launch_row_copies(const RowCopies &c, bool to_dense, hipStream_t st);

// The wave kernels (AttnConfig::wave): forward, and dQ then dK/dV.
int launch_fwd_wave(const FwdArgs &a, hipStream_t st);
int launch_bwd_wave(const BwdArgs &a, hipStream_t st);

}  // namespace attn
}  // namespace pb
