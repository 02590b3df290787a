// Gated activation feeding the row-split down projection: act[r, i] = silu(gu[r, i]) * gu[r, inter + i], bf16.
//
// This is the producer of the tree matmul's X operand (the MLP of the reference's models runs vLLM's
// SiluAndMul between the merged gate/up projection and down_proj, whose forward is the patched
// RowParallelLinear, src/patch/patch_tp_invariant.py:10-48).  Arithmetic: silu in fp32, rounded to bf16,
// then the product rounded to bf16 -- two roundings, as an unfused `F.silu(gate) * up` on bf16 tensors
// gives.  Elementwise, so batch invariant by construction.  HBM bound: 6 bytes per output element.
#include "common.h"
#include "qk_norm_rope.h"
#include "silu_mul.h"

namespace tbik {


// One thread per 8 outputs (16-byte loads and stores); 2-D grid-stride over (row, pack).
template <bool F16>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu, int64_t ld_in,
                                                       uint16_t* __restrict__ out, int64_t ld_out, int64_t rows,
                                                       int packs_per_row, int inter) {
  const int64_t total = rows * packs_per_row;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    const int64_t r = i / packs_per_row;
    const int c = (int)(i - r * packs_per_row) * 8;
    const uint4 g = *reinterpret_cast<const uint4*>(gu + r * ld_in + c);
    const uint4 u = *reinterpret_cast<const uint4*>(gu + r * ld_in + inter + c);
    uint4 o;
    o.x = silu_mul_pair<F16>(g.x, u.x);
    o.y = silu_mul_pair<F16>(g.y, u.y);
    o.z = silu_mul_pair<F16>(g.z, u.z);
    o.w = silu_mul_pair<F16>(g.w, u.w);
    *reinterpret_cast<uint4*>(out + r * ld_out + c) = o;
  }
}

int silu_mul_dispatch(const void* gate_up, int64_t ld_in, void* out, int64_t ld_out, int64_t rows, int inter, bool f16,
                      hipStream_t stream) {
  if (rows < 0 || inter <= 0 || ld_in < 2 * (int64_t)inter || ld_out < inter) return TBIK_ERR_INVALID;
  if (rows == 0 && !(inter & 7)) return TBIK_OK;
  if (!gate_up || !out) return TBIK_ERR_INVALID;
  if ((inter & 7) || (ld_in & 7) || (ld_out & 7)) return TBIK_ERR_ALIGNMENT;
  if ((reinterpret_cast<uintptr_t>(gate_up) & 15) || (reinterpret_cast<uintptr_t>(out) & 15)) return TBIK_ERR_ALIGNMENT;
  if (rows == 0) return TBIK_OK;
  const int packs = inter / 8;
  const int64_t blocks = (rows * packs + 255) / 256;
  const unsigned grid = (unsigned)(blocks < 16384 ? blocks : 16384);
  if (f16)
    hipLaunchKernelGGL(silu_mul_kernel<true>, dim3(grid), dim3(256), 0, stream, static_cast<const uint16_t*>(gate_up), ld_in,
                       static_cast<uint16_t*>(out), ld_out, rows, packs, inter);
  else
    hipLaunchKernelGGL(silu_mul_kernel<false>, dim3(grid), dim3(256), 0, stream, static_cast<const uint16_t*>(gate_up), ld_in,
                       static_cast<uint16_t*>(out), ld_out, rows, packs, inter);
  return hip_code(hipGetLastError());
}

}  // namespace tbik

namespace tbik {

// ------------------------------------------------------------------------------------------------
// Per-head q/k RMSNorm + rotary embedding + KV-cache write for a Qwen3-style attention block, from the fused qkv projection
// output [tokens, (Hq + 2*Hkv) * 128]:
//   query heads : q_out[token, h, :]          = rope(rmsnorm(q) * q_weight)
//   key heads   : k_cache[seq, h, pos, :]      = rope(rmsnorm(k) * k_weight)
//   value heads : vt_cache[seq, h, :, pos]     = v                    (the attention kernel reads V transposed)
// rmsnorm as in rmsnorm_kernel (fp32 statistics, the normalised value rounded to bf16, then a bf16 multiply by the
// weight); rope is rotate-half in fp32 with angle pos * inv_freq[i], rounded once to bf16.  Everything is per
// (token, head): batch invariant by construction.  Lane l owns channels l and l + 64 (a rotary pair).
// This is the caller side of the fixed-order attention (the reference patches vLLM's rotary embedding and leaves the
// rest to the engine, src/patch/patch_training_inference_align.py:35-44).
//
// Bound: memory (12 KiB in and out per token at 32/8 heads) once two things are out of its way.  Sine and cosine belong
// to the token, not to the head: a wavefront takes HPW heads of one token and forms them once (formed per head they kept
// the vector units busy three times as long as the memory).  And the transposed values: stored by the wavefront of a
// token they are 2-byte pieces max_len apart, so work-groups of 64 tokens x one value head pass them through LDS and
// store, per channel, what consecutive tokens leave at consecutive positions.  9,096 tokens of three prompts: 132 -> 47 us
// (a copy of the bytes takes 44), 1000 tokens 17.3 -> 9.1, a few tokens 5 as before.
// ------------------------------------------------------------------------------------------------
struct QkRopeArgs {
  const uint16_t* qkv;
  int64_t ld;
  const uint16_t* qw;
  const uint16_t* kw;
  const float* inv_freq;   // [64]
  const int64_t* pos;      // [tokens]
  const int64_t* seq;      // [tokens]
  uint16_t* q_out;         // [tokens, Hq, 128]
  uint16_t* k_cache;       // [B, Hkv, L, 128]
  uint16_t* vt_cache;      // [B, Hkv, 128, L]
  int64_t tokens;
  int q_heads, kv_heads, max_len, batch;
  float eps;
};

constexpr int VT_TOKENS = 64;   // tokens per work-group of the value part

// Work-groups [0, value_groups): 64 tokens of one value head each; the others: four wavefronts of HPW query or key heads.
constexpr int HPW = 8;   // heads per wavefront (1, 2, 4: 103, 69, 54 us at 9,096 tokens; no difference below 200)

__global__ __launch_bounds__(256) void qk_norm_rope_cache_kernel(const QkRopeArgs a, int value_groups, int q_units, int units) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((int)blockIdx.x < value_groups) {
    __shared__ uint16_t tile[VT_TOKENS][130];   // rows an odd number of words apart: a column is free of bank conflicts
    const int h = blockIdx.x % a.kv_heads;
    const int64_t t0 = (int64_t)(blockIdx.x / a.kv_heads) * VT_TOKENS;
    const uint16_t* src = a.qkv + t0 * a.ld + (int64_t)(a.q_heads + a.kv_heads + h) * 128;
    const int nt = (int)(a.tokens - t0 < VT_TOKENS ? a.tokens - t0 : VT_TOKENS);
#pragma unroll
    for (int i = 0; i < VT_TOKENS / 4; i++) {   // wavefront w: tokens w, w + 4, ..., two channels per lane
      const int t = min(i * 4 + wave, nt - 1);
      uint16_t lo = src[t * a.ld + 2 * lane], hi = src[t * a.ld + 2 * lane + 1];
      *reinterpret_cast<uint32_t*>(&tile[i * 4 + wave][2 * lane]) = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    __syncthreads();
    if (lane >= nt) return;
    const int64_t pos = a.pos[t0 + lane], sq = a.seq[t0 + lane];
    if (sq < 0 || sq >= a.batch || pos < 0 || pos >= a.max_len) return;
    uint16_t* dst = a.vt_cache + ((sq * a.kv_heads + h) * 128 + wave * 32) * (int64_t)a.max_len + pos;
#pragma unroll 8
    for (int c = 0; c < 32; c++) dst[(int64_t)c * a.max_len] = tile[lane][wave * 32 + c];
    return;
  }
  const int64_t unit = (int64_t)(blockIdx.x - value_groups) * 4 + wave;
  const int64_t tok = unit / units;
  if (tok >= a.tokens) return;
  const int u = (int)(unit % units);
  const bool is_q = u < q_units;
  const int h0 = (is_q ? u : u - q_units) * HPW;
  const int nh = min(HPW, (is_q ? a.q_heads : a.kv_heads) - h0);
  const uint16_t* src = a.qkv + tok * a.ld + (int64_t)((is_q ? 0 : a.q_heads) + h0) * 128;
  uint16_t r1[HPW], r2[HPW];
#pragma unroll
  for (int i = 0; i < HPW; i++) {   // all heads of the wavefront are in flight while sine and cosine are formed
    const int o = min(i, nh - 1) * 128;
    r1[i] = src[o + lane];
    r2[i] = src[o + lane + 64];
  }
  const uint16_t* w = is_q ? a.qw : a.kw;
  const float w1 = bf16_bits_to_f32(w[lane]), w2 = bf16_bits_to_f32(w[lane + 64]);
  const int64_t pos = a.pos[tok];
  uint16_t* dst;
  int64_t step;
  if (is_q) {
    dst = a.q_out + (tok * a.q_heads + h0) * 128;
    step = 128;
  } else {
    const int64_t sq = a.seq[tok];
    if (sq < 0 || sq >= a.batch || pos < 0 || pos >= a.max_len) return;
    dst = a.k_cache + (((sq * a.kv_heads + h0) * (int64_t)a.max_len) + pos) * 128;
    step = (int64_t)a.max_len * 128;
  }
  const RopeFactors rope(pos, a.inv_freq, lane);
#pragma unroll
  for (int i = 0; i < HPW; i++) {
    if (i >= nh) break;
    const uint32_t o = qk_norm_rope_head(r1[i], r2[i], w1, w2, rope, a.eps);
    dst[i * step + lane] = (uint16_t)(o & 0xffffu);
    dst[i * step + lane + 64] = (uint16_t)(o >> 16);
  }
}

int qk_norm_rope_cache_dispatch(const void* qkv, int64_t ld, const void* q_weight, const void* k_weight,
                                const float* inv_freq, const int64_t* positions, const int64_t* seq_of_token, void* q_out,
                                void* k_cache, void* vt_cache, int64_t tokens, int q_heads, int kv_heads, int head_dim,
                                int max_len, int batch, float eps, hipStream_t stream) {
  if (!qkv || !q_weight || !k_weight || !inv_freq || !positions || !seq_of_token || !q_out || !k_cache || !vt_cache)
    return TBIK_ERR_INVALID;
  if (tokens < 0 || q_heads <= 0 || kv_heads <= 0 || max_len <= 0 || batch <= 0) return TBIK_ERR_INVALID;
  if (head_dim != 128) return TBIK_ERR_UNSUPPORTED;
  if (ld < (int64_t)(q_heads + 2 * kv_heads) * 128) return TBIK_ERR_INVALID;
  if (tokens == 0) return TBIK_OK;
  QkRopeArgs a{static_cast<const uint16_t*>(qkv), ld, static_cast<const uint16_t*>(q_weight),
               static_cast<const uint16_t*>(k_weight), inv_freq, positions, seq_of_token, static_cast<uint16_t*>(q_out),
               static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(vt_cache), tokens, q_heads, kv_heads, max_len, batch, eps};
  const int q_units = (q_heads + HPW - 1) / HPW, units = q_units + (kv_heads + HPW - 1) / HPW;
  const int64_t vg = (tokens + VT_TOKENS - 1) / VT_TOKENS * kv_heads, blocks = vg + (tokens * units + 3) / 4;
  if (blocks > 0x7fffffff) return TBIK_ERR_INVALID;
  hipLaunchKernelGGL(qk_norm_rope_cache_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a, (int)vg, q_units, units);
  return hip_code(hipGetLastError());
}

}  // namespace tbik
