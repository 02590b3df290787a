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
// token they are 2-byte pieces max_len apart, so work-groups of 64 tokens x 128 / VS channels of a value head pass them
// through LDS and store, per channel, what consecutive tokens leave at consecutive positions.  9,096 tokens of three
// prompts: 132 -> 47 us (a copy of the bytes takes 44).  A call of fewer tokens is a chain of latencies and of stores that
// may all be scattered (one new token for each of many sequences), and takes smaller pieces; see the dispatch.
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

// Work-groups [0, value_groups): 64 tokens of 128 / VS channels of one value head each; the others: four wavefronts of HPW
// query or key heads.
template <int VS, int HPW>
__global__ __launch_bounds__(256) void qk_norm_rope_cache_kernel(const QkRopeArgs a, int value_groups, int q_units, int units) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((int)blockIdx.x < value_groups) {
    constexpr int NC = 128 / VS, PAIRS = NC / 2;   // channels of the work-group
    __shared__ uint16_t tile[VT_TOKENS][NC + 2];   // rows an odd number of words apart: a column is free of bank conflicts
    const int unit = blockIdx.x / VS, c0 = blockIdx.x % VS * NC;
    const int h = unit % a.kv_heads;
    const int64_t t0 = (int64_t)(unit / a.kv_heads) * VT_TOKENS;
    const uint16_t* src = a.qkv + t0 * a.ld + (int64_t)(a.q_heads + a.kv_heads + h) * 128 + c0;
    const int nt = (int)(a.tokens - t0 < VT_TOKENS ? a.tokens - t0 : VT_TOKENS);
#pragma unroll
    for (int i = 0; i < VT_TOKENS * PAIRS / 256; i++) {   // two channels of a token per thread
      const int e = i * 256 + threadIdx.x, row = e / PAIRS, c = 2 * (e % PAIRS);
      const int t = min(row, nt - 1);
      uint16_t lo = src[t * a.ld + c], hi = src[t * a.ld + c + 1];
      *reinterpret_cast<uint32_t*>(&tile[row][c]) = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    __syncthreads();
    if (lane >= nt) return;
    const int64_t pos = a.pos[t0 + lane], sq = a.seq[t0 + lane];
    if (sq < 0 || sq >= a.batch || pos < 0 || pos >= a.max_len) return;
    uint16_t* dst = a.vt_cache + ((sq * a.kv_heads + h) * 128 + c0 + wave * (NC / 4)) * (int64_t)a.max_len + pos;
#pragma unroll 8
    for (int c = 0; c < NC / 4; c++) dst[(int64_t)c * a.max_len] = tile[lane][wave * (NC / 4) + c];
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

template <int VS, int HPW>
static int qk_rope_launch(const QkRopeArgs& a, hipStream_t stream) {
  const int q_units = (a.q_heads + HPW - 1) / HPW, units = q_units + (a.kv_heads + HPW - 1) / HPW;
  const int64_t vg = (a.tokens + VT_TOKENS - 1) / VT_TOKENS * a.kv_heads * VS, blocks = vg + (a.tokens * units + 3) / 4;
  if (blocks > 0x7fffffff) return TBIK_ERR_INVALID;
  hipLaunchKernelGGL((qk_norm_rope_cache_kernel<VS, HPW>), dim3((unsigned)blocks), dim3(256), 0, stream, a, (int)vg, q_units, units);
  return hip_code(hipGetLastError());
}
// Heads per wavefront: by the (token, head) pairs there are, so that they still occupy the chip.  us of one launch in a graph
// at 32/8 heads, 1, 2, 4, 8 heads (a wavefront and value per token and head before): 1 token 2.4, 2.5, 2.9, 3.7 (2.2);
// 64 tokens of one prompt 2.9, 2.8, 3.2, 4.0 (2.9); 256 5.1, 4.2, 4.1, 4.7 (6.2); 1000 13.5, 10.1, 8.7, 8.6 (16.1).
template <int VS>
static int qk_rope_by_heads(const QkRopeArgs& a, hipStream_t stream) {
  const int64_t pairs = a.tokens * (a.q_heads + a.kv_heads);
  if (pairs <= 2048) return qk_rope_launch<VS, 1>(a, stream);
  if (pairs <= 8192) return qk_rope_launch<VS, 2>(a, stream);
  if (pairs <= 32768) return qk_rope_launch<VS, 4>(a, stream);
  return qk_rope_launch<VS, 8>(a, stream);
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
  // Channels per work-group of the values, for stores that are scattered: sequences with one token each at 8 KV heads,
  // VS = 1, 4, 16 (before): 64 of them 11.7, 4.9, 3.5 us (3.9), 200 10.7, 6.7, 6.3 (6.0), 400 12.1, 9.6, 10.3 (9.8); 200 at 16
  // KV heads 13.0, 8.3, 9.3 (7.6).  A prompt of 2000 tokens 14.1, 15.4, 19.9 (30.9).
  const int64_t tiles = (tokens + VT_TOKENS - 1) / VT_TOKENS * kv_heads;
  if (tiles <= 32) return qk_rope_by_heads<16>(a, stream);
  if (tiles < 256) return qk_rope_by_heads<4>(a, stream);
  return qk_rope_by_heads<1>(a, stream);
}

}  // namespace tbik
