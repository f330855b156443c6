// Sum of a row held by a whole workgroup (the *_wide norm kernels).
#pragma once

#include "common.hpp"
#include "lds_dma.hpp"

namespace pb {

// One value per lane summed over the workgroup, through LDS with one barrier;
// callers take the two slots in turn, so a wave never overwrites a sum another
// wave is still reading.  The barrier has no memory fence: loads issued before
// it stay in flight.  The waves' sums are added pairwise: one after the other,
// 16 of them would round more than the one-wave kernel's sum (fp32 [1000,
// 12288], y against float64 5.97e-8 there, 6.43e-8 in sequence, 5.77e-8 pairwise).
template <int THREADS>
__device__ __forceinline__ float row_sum(float v, float (*red)[THREADS / 64], int slot) {
  constexpr int W = THREADS / 64;
  v = wave_sum_full(v);
  if ((threadIdx.x & 63) == 0) red[slot][threadIdx.x >> 6] = v;
  __builtin_amdgcn_s_waitcnt(0xC07F);  // the LDS write is done (lgkmcnt(0))
  block_sync_nofence();
  float s[W];
#pragma unroll
  for (int k = 0; k < W; ++k) s[k] = red[slot][k];
#pragma unroll
  for (int n = W / 2; n >= 1; n /= 2)
#pragma unroll
    for (int k = 0; k < n; ++k) s[k] += s[k + n];
  return s[0];
}

}  // namespace pb
