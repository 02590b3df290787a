// Per-head RMSNorm + rotary embedding of ONE head (128 channels) by ONE wavefront, shared by the stand-alone kernel
// (elementwise.hip) and by the decode attention kernel that forms its own queries and the new key (attention.hip): one
// body, so both give the same bits.
//
// Lane l owns channels l and l + 64 (a rotary pair).  rmsnorm as in rmsnorm_row.h (fp32 statistics, the normalised
// value rounded to bf16, then a bf16 multiply by the weight); rope is rotate-half in fp32 with angle pos * inv_freq[l],
// rounded once to bf16.  Returns the two results packed (channel l in the low half, l + 64 in the high half).
#pragma once
#include "common.h"

namespace tbik {

// The rotation of the pair (l, l + 64) at position `pos`: one per token, whatever the head.
struct RopeFactors {
  float c, s;
  __device__ __forceinline__ RopeFactors(int64_t pos, const float* inv_freq, int lane) {
#pragma clang fp contract(off)
    const float ang = (float)pos * inv_freq[lane];
    c = cosf(ang), s = sinf(ang);
  }
};

__device__ __forceinline__ uint32_t qk_norm_rope_head(uint16_t r1, uint16_t r2, float w1, float w2, const RopeFactors& rope, float eps) {
  // every product and sum is rounded on its own, except where a fused multiply-add is written out: left to the
  // compiler, a multiplication could be fused with the next addition in one kernel and not in the other
#pragma clang fp contract(off)
  const float x1 = bf16_bits_to_f32(r1), x2 = bf16_bits_to_f32(r2);
  const float ss = wave_sum(__builtin_fmaf(x1, x1, x2 * x2));
  const float rs = 1.0f / sqrtf(ss * (1.0f / 128.0f) + eps);
  const uint32_t nrm = pack_bf16x2(x1 * rs, x2 * rs);
  const uint32_t wv = pack_bf16x2(bf16_lo(nrm) * w1, bf16_hi(nrm) * w2);
  const float y1 = bf16_lo(wv), y2 = bf16_hi(wv);
  return pack_bf16x2(y1 * rope.c - y2 * rope.s, y2 * rope.c + y1 * rope.s);
}

__device__ __forceinline__ uint32_t qk_norm_rope_head(uint16_t r1, uint16_t r2, const uint16_t* w, int64_t pos,
                                                      const float* inv_freq, float eps, int lane) {
  const float w1 = bf16_bits_to_f32(w[lane]), w2 = bf16_bits_to_f32(w[lane + 64]);
  return qk_norm_rope_head(r1, r2, w1, w2, RopeFactors(pos, inv_freq, lane), eps);
}

}  // namespace tbik
