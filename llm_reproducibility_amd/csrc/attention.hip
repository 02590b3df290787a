// Fixed-order causal attention for gfx950 (bf16, head_dim 128, grouped-query heads).  A query row is always the four
// lanes {j, j+16, j+32, j+48} of one wavefront; three kernels differ in what else the wavefront and its work-group hold:
//   attention_kernel        one wavefront per (16 consecutive queries of a sequence, query head), operands from global
//                           memory (any cache length);
//   attention_group_kernel  the G query heads of a KV head times one or two blocks of 16 queries in the wavefronts of a
//                           work-group, keys and values staged in LDS once for all of them (prefill and chunked prefill);
//   attention_decode_kernel the few new queries of a sequence times the G heads as the 16 rows of ONE tile, the output
//                           channels split over four wavefronts, four more wavefronts bringing the tiles in (decode).
//
// Counterpart of the reference's fixed-tile attention for train/inference alignment
// (_kernel_unified_attention_2d, src/patch/patch_training_inference_align.py:171-487: one pass over the
// keys in tiles of 32, online softmax, no split over the key axis, the same kernel for prefill and decode).
//
// Invariance argument: a query row is owned by the four lanes {j, j+16, j+32, j+48}; its scores, its
// running maximum / denominator and its output accumulators never mix with another row's.  The keys are cut into
// chunks of 512 at fixed positions.  Inside a chunk they are visited in ascending tiles of 32, starting from an empty
// state (reference point, denominator, accumulators), whatever the batch or the block looks like; a tile that lies
// entirely behind a row's causal horizon contributes exp(-inf) = 0 and a rescale by exactly 1.0, so the number of
// tiles the BLOCK walks does not change the row.  The chunks' states are merged in ascending order (merge_chunk),
// those behind a row's horizon left out.  Prefill (16 rows per block) and decode (1 valid row)
// therefore produce the same bits for the same token, and heads can be sharded freely; and because no chunk waits for
// another, a few sequences with long contexts spread their chunks over the chip.
//
// Layouts: q/out [tokens, q_heads, 128]; K cache [batch, kv_heads, max_len, 128]; V cache TRANSPOSED
// [batch, kv_heads, 128, max_len] so that the P*V MFMA operand (8 consecutive keys of one channel) is a
// contiguous load.  Cache entries behind ctx_len must be finite (they are multiplied by an exact 0).
#include "common.h"
#include "lds_direct.h"
#include "qk_norm_rope.h"

namespace tbik {

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k_cache;
  const uint16_t* vt_cache;
  uint16_t* out;
  const int* q_start;  // [batch] first token row of the sequence in q/out
  const int* q_len;    // [batch] new tokens of the sequence
  const int* ctx_len;  // [batch] keys visible to the LAST new token (cache length including the new tokens)
  int q_heads, kv_heads, max_len;
  float scale_log2;    // log2(e) / sqrt(head_dim): scores are kept in the base-2 domain
};

constexpr int HD = 128;
constexpr int CHUNK_TILES = 16;           // key tiles per chunk: 512 keys
constexpr float kNoKey = -__FLT_MAX__;    // reference point of an empty state: no finite score lies below it (see move_reference)

// Where the chunks of a row go when different work-groups compute them (SPLIT): slot (sequence * q_rows + query) *
// q_heads + head of [nchunks] states.  q_rows are the queries per sequence that the kernels' tiles have room for and not
// the caller's max_q_len: they compute every row that the device's q_len says there is, up to those.
struct SplitArgs {
  float* o;      // [slot][nchunks][128] accumulators
  float* ml;     // [slot][nchunks][2] reference point, denominator
  int nchunks;   // chunks of the cache length
  int q_rows;
};

// The decode kernel that forms its own queries and the new key/value (FUSED): sequence b's one new token is row b of the
// fused qkv projection output, at position ctx_len[b] - 1.
struct QkvArgs {
  const uint16_t* qkv;    // [batch, (q_heads + 2 kv_heads) * 128], row stride ld
  int64_t ld;
  const uint16_t* qw;     // per-head q norm weight [128]
  const uint16_t* kw;     // per-head k norm weight [128]
  const float* inv_freq;  // [64]
  uint16_t* k_cache;      // the caches of AttnArgs, writable: the new key and value are filed here as well
  uint16_t* vt_cache;
  float eps;
};

// One online-softmax update of a query row for a tile of 32 keys, in the pieces that the kernels of this file put together (the
// same bits in all).  Row 4g + i of the 16-row sub-tile u of a key tile is key 8g + 4u + i (key_row), so lane (j, g) holds the
// scores of query j for the eight consecutive keys k0 + 8g .. +7 in s[0], s[1], and its probabilities are the B operand of a
// P*V MFMA whose A operand is eight consecutive keys of a channel: 16 bytes of the V^T cache as they lie.
// Every product and sum below is rounded on its own, except where a fused multiply-add is written out: left to the
// compiler, a multiplication could be fused with the next addition in one instantiation and not in another, and the
// kernels would no longer agree bit for bit.
__device__ __forceinline__ int key_row(int u, int r) { return 8 * (r >> 2) + 4 * u + (r & 3); }

// the causal mask (needed only for tiles that reach beyond some row's horizon; the others' values do not change)
__device__ __forceinline__ void mask_scores(f32x4 (&s)[2], int k0, int g, int qpos) {
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int i = 0; i < 4; i++) s[u][i] = (k0 + 8 * g + 4 * u + i <= qpos) ? s[u][i] : -INFINITY;
}
// The largest of the lane's eight raw scores; scaled, it is the largest of the scaled ones (the scale is positive and
// rounding is monotonic).  NaN-propagating: a NaN score makes the row NaN, as it would through the sum.
__device__ __forceinline__ float lane_max(const f32x4 (&s)[2]) {
  return LaneMaxNaN::f(LaneMaxNaN::f(LaneMaxNaN::f(s[0][0], s[0][1]), LaneMaxNaN::f(s[0][2], s[0][3])),
                       LaneMaxNaN::f(LaneMaxNaN::f(s[1][0], s[1][1]), LaneMaxNaN::f(s[1][2], s[1][3])));
}
// The reference point of the exponentials moves lazily: only when a score of this tile exceeds it by more than 2^kLazy
// (probabilities then stay below 2^kLazy instead of 1: no loss in fp32 sums or in the relative precision of a bf16
// probability, and out = o / l is the same quotient).  After the first tiles of a chunk it practically never moves.  The rule
// looks at a row's own scores in its fixed tile order only, so it is the same for prefill, chunked prefill and decode; and
// while no lane of a wavefront has a score that far up (score_exceeds), move_reference would leave every row where it is
// and return exactly 1.0 -- the grouped kernel asks that first and skips the exchange between a row's lanes, the
// exponential and the rescale.
// A row's first key of a chunk moves it from kNoKey to a score; in a tile that lies entirely behind the horizon it stays
// where it is (kNoKey is finite, so kNoKey - kNoKey is 0 and not NaN) and every probability is 2^-inf = 0.
constexpr float kLazy = 8.0f;
__device__ __forceinline__ bool score_exceeds(float lmax, float scale_log2, float m) {
#pragma clang fp contract(off)
  return lmax * scale_log2 > m + kLazy;
}
// returns the factor for the row's accumulators and (applied here) denominator
__device__ __forceinline__ float move_reference(float lmax, float scale_log2, float& m, float& l) {
#pragma clang fp contract(off)
  float tmax = xor_step<16, LaneMaxNaN>(lmax);
  tmax = xor_step<32, LaneMaxNaN>(tmax);
  const float cand = tmax * scale_log2;
  const float m_new = cand > m + kLazy ? cand : m;
  const float alpha = __builtin_amdgcn_exp2f(m - m_new);        // exactly 1.0 when the reference point did not move
  m = m_new;
  l = l * alpha;
  return alpha;
}
// The lane's eight probabilities, 2^(score * scale - m) as one fused multiply-add and one hardware exponential each (the
// arguments are <= kLazy, and a result below 2^-126 is dropped, which neither the denominator nor a bf16 probability can
// show).  The denominator is kept per lane and summed over a row's four lanes where a chunk ends (row_sum).
__device__ __forceinline__ bf16x8 probabilities(const f32x4 (&s)[2], float scale_log2, float m, float& l) {
#pragma clang fp contract(off)
  float pv[8];
#pragma unroll
  for (int e = 0; e < 8; e++) pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e >> 2][e & 3], scale_log2, -m));
  l = l + (((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7])));
  return __builtin_bit_cast(bf16x8, u32x4{pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3]), pack_bf16x2(pv[4], pv[5]),
                                          pack_bf16x2(pv[6], pv[7])});
}
__device__ __forceinline__ float row_sum(float l) { return xor_step<32, LaneSum>(xor_step<16, LaneSum>(l)); }

// The merge of a row's next chunk (m, l, and below each accumulator) into its state so far (M, L): both are brought to the
// larger reference point, rounded as written in every kernel (no contraction).
__device__ __forceinline__ void merge_chunk(float& M, float& L, float m, float l, float& fa, float& fb) {
#pragma clang fp contract(off)
  const float top = LaneMaxNaN::f(M, m);
  fa = __builtin_amdgcn_exp2f(M - top);
  fb = __builtin_amdgcn_exp2f(m - top);
  M = top;
  L = __builtin_fmaf(L, fa, l * fb);
}
__device__ __forceinline__ float merge_acc(float O, float fa, float o, float fb) {
#pragma clang fp contract(off)
  return __builtin_fmaf(O, fa, o * fb);
}

__global__ __launch_bounds__(64) void attention_kernel(const AttnArgs a) {
  const int b = blockIdx.z;
  const int h = blockIdx.y;
  const int qb = blockIdx.x;
  const int qlen = a.q_len[b];
  if (qb * 16 >= qlen) return;
  const int lane = threadIdx.x;
  const int j = lane & 15;   // query row inside the block (also: key row of a K fragment, channel row of a V fragment)
  const int g = lane >> 4;   // lane group: which 8-wide k slice of an MFMA operand, which 4 rows of an MFMA result
  const int ctx = a.ctx_len[b];
  const int kvh = h / (a.q_heads / a.kv_heads);
  const int qrow = qb * 16 + j;                     // row inside the sequence's new tokens
  const bool qvalid = qrow < qlen;
  const int qpos = ctx - qlen + min(qrow, qlen - 1);  // absolute position of this lane's query
  const int last_pos = ctx - qlen + min(qb * 16 + 15, qlen - 1);

  // Q as the MFMA "B" operand: lane (j, g) holds q[j][32c + 8g .. +7] for the four 32-wide channel chunks c
  const uint16_t* qp = a.q + ((int64_t)(a.q_start[b] + min(qrow, qlen - 1)) * a.q_heads + h) * HD;
  bf16x8 qf[4];
#pragma unroll
  for (int c = 0; c < 4; c++) qf[c] = *reinterpret_cast<const bf16x8*>(qp + c * 32 + g * 8);

  const uint16_t* kbase = a.k_cache + ((int64_t)b * a.kv_heads + kvh) * a.max_len * HD;
  const uint16_t* vbase = a.vt_cache + ((int64_t)b * a.kv_heads + kvh) * (int64_t)HD * a.max_len;

  f32x4 o[8];  // output accumulators, transposed: lane (j, g) holds out[j][16t + 4g .. +3] for the channel tiles t
#pragma unroll
  for (int t = 0; t < 8; t++) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNoKey;     // reference point of the exponentials (base-2 domain; a lazily updated running maximum), identical in the four lanes of a row
  float l = 0.f;        // running denominator
  f32x4 ot[8];          // the merged chunks so far
  float mt = 0.f, lt = 0.f;
  // chunk `c` is complete: merged into the rows that see it, and an empty state for the next
  auto end_chunk = [&](int c) {
    l = row_sum(l);
    if (c == 0) {
      mt = m, lt = l;
#pragma unroll
      for (int t = 0; t < 8; t++) ot[t] = o[t];
    } else if (qpos >= c * CHUNK_TILES * 32) {
      float fa, fb;
      merge_chunk(mt, lt, m, l, fa, fb);
#pragma unroll
      for (int t = 0; t < 8; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) ot[t][i] = merge_acc(ot[t][i], fa, o[t][i], fb);
    }
    m = kNoKey, l = 0.f;
#pragma unroll
    for (int t = 0; t < 8; t++) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  };

  const int ntiles = last_pos / 32 + 1;
  for (int tile = 0; tile < ntiles; tile++) {
    const int k0 = tile * 32;
    if (tile != 0 && tile % CHUNK_TILES == 0) end_chunk(tile / CHUNK_TILES - 1);
    // ---- scores: two sub-tiles of 16 keys; lane (j, g) receives keys k0 + 8g + 4u + i of query j
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int krow = min(k0 + key_row(u, j), a.max_len - 1);
      const uint16_t* kp = kbase + (int64_t)krow * HD + g * 8;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kp + c * 32);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[c], acc, 0, 0, 0);
      }
      s[u] = acc;
    }
    mask_scores(s, k0, g, qpos);
    const float alpha = move_reference(lane_max(s), a.scale_log2, m, l);
    const bf16x8 pf = probabilities(s, a.scale_log2, m, l);
    // ---- out^T += V^T * P: "A" operand lane (j, g) holds channel 16t + j, the same 8 keys
    const int kv0 = min(k0 + 8 * g, a.max_len - 4);
    const int kv1 = min(k0 + 8 * g + 4, a.max_len - 4);
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const uint16_t* vp = vbase + (int64_t)(16 * t + j) * a.max_len;
      const uint2 va = *reinterpret_cast<const uint2*>(vp + kv0);
      const uint2 vb = *reinterpret_cast<const uint2*>(vp + kv1);
      const bf16x8 vf = __builtin_bit_cast(bf16x8, u32x4{va.x, va.y, vb.x, vb.y});
      f32x4 scaled = {o[t][0] * alpha, o[t][1] * alpha, o[t][2] * alpha, o[t][3] * alpha};
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, scaled, 0, 0, 0);
    }
  }
  end_chunk((ntiles - 1) / CHUNK_TILES);
  if (!qvalid) return;
  const float inv = 1.0f / lt;
  uint16_t* op = a.out + ((int64_t)(a.q_start[b] + qrow) * a.q_heads + h) * HD;
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const uint32_t lo = pack_bf16x2(ot[t][0] * inv, ot[t][1] * inv);
    const uint32_t hi = pack_bf16x2(ot[t][2] * inv, ot[t][3] * inv);
    *reinterpret_cast<uint2*>(op + 16 * t + 4 * g) = make_uint2(lo, hi);
  }
}

// Key tiles in LDS.  A direct load puts lane l's 16 bytes at (wave-uniform address) + 16 l, so the layout is made on the global
// side: each lane fetches the 16-byte chunk that belongs at its place.
//   K rows [keys][256 bytes]: position pc of key row kr holds chunk pc ^ k_swizzle(kr);
//   V^T rows [128 channels][128 bytes = 64 keys]: position pc of channel row r holds chunk pc ^ v_swizzle(r).
// A 16-byte read is served for lanes {0-7, 16-23} together (then {8-15, 24-31}, ...): the eight rows and two neighbouring
// chunks of such a pass cover all 64 banks in both.
__device__ __forceinline__ int k_swizzle(int kr) { return 2 * ((kr & 3) + 4 * ((kr >> 3) & 1)); }
__device__ __forceinline__ int v_swizzle(int r) { return 2 * ((r >> 1) & 3); }
// byte offsets of lane (j, g)'s fragments: chunk c of key key_row(0, j) (sub-tile 1 lies four rows = 1024 bytes on), and chunk c
// = eight keys of channel row j (sixteen channels are 16 rows on)
__device__ __forceinline__ uint32_t k_fragment(int j, int c) { return key_row(0, j) * 256 + ((c ^ k_swizzle(key_row(0, j))) << 4); }
__device__ __forceinline__ uint32_t v_fragment(int j, int c) { return j * 128 + ((c ^ v_swizzle(j)) << 4); }

// ------------------------------------------------------------------------------------------------
// Grouped variant: one work-group of NW = G * WQ wavefronts per (16 * QB * WQ consecutive queries, KV head, sequence).  A
// wavefront holds one of the G query heads that share the KV head and QB blocks of 16 queries; the keys are brought in 64 at
// a time (K and V^T, 32 KiB) by direct loads into an LDS ring of NS slots, once for the whole work-group, and every fragment
// read from there serves the wavefront's QB blocks.  NLD > 0: that many more wavefronts do all the loading (their scalar
// address arithmetic and the loads are a third of a tile's instructions) and none of the computing.  A row's arithmetic -- the
// lanes that own it, the MFMA chain, the order of the softmax updates -- is exactly that of attention_kernel above, so the kernels
// produce the same bits.
// SPLIT_CHUNKS: a work-group takes one chunk of the keys (blockIdx.z) and leaves its state in the workspace for
// attention_merge_kernel: a few new tokens against a long cache are a handful of work-groups otherwise.
// What bounds it: vector issue and matrix pipes together.  8192 tokens of 32 heads on two blocks (503 us, 1.09 PFLOP/s; 599 before):
// per 32 queries x 32 keys of a wavefront 512 cycles of MFMA (busy 51 % of the SIMD's cycles), some 100 vector instructions
// and 16 exponentials (47 %), no bank conflict, the LDS read port busy a quarter of the time.  One fragment read per 16
// queries made it the LDS and the L2 (a 64-byte half of a V^T line per load and tile: 8.4 TB/s) instead; in work-groups of
// 64 queries, which halve the key traffic once more, it takes the same time (532), and so does forming a tile's scores ahead.
// Launches that leave CUs short of work-groups are a chain of tiles, 0.53 us each and 0.39 with loaders beside them.
// (Two vector instructions per MFMA issue behind it, each further one costs its 1.8 ns: on one CU 7.15 / 7.67 / 9.31 / 11.31 ns per MFMA
// with 0 / 2 / 3 / 4 FMAs on two wavefronts per SIMD, 7.86 / 9.21 / 10.84 / 12.69 on one; on all 256 the clock pays for them, 8.10 /
// 10.15 / 11.92 / 14.26.  A tile has three and half an exponential, so work moves the time only where it goes away: scores a tile
// ahead, and two blocks' exponentials between each other's MFMAs, were level.)
// ------------------------------------------------------------------------------------------------
// chunks: the cache has a single one / a work-group walks them all / a work-group takes one
enum { ONE_CHUNK, ALL_CHUNKS, SPLIT_CHUNKS };
constexpr int UNIT = 64, UNIT_BYTES = 4 * UNIT * HD;  // keys of a ring slot; 16 KiB of K, 16 KiB of V^T
template <int G, int WQ, int QB, int NS, int CHUNKS, int NLD>
__global__ __launch_bounds__(64 * (G * WQ + NLD), QB == 2 || G * WQ == 8 ? 2 : 1) void attention_group_kernel(const AttnArgs a, const SplitArgs sp) {
  constexpr bool SPLIT = CHUNKS == SPLIT_CHUNKS;
  constexpr int NW = G * WQ, ROWS = 16 * QB * WQ;
  constexpr int NL = NLD ? NLD : NW;                    // wavefronts that load
  constexpr int PI = 16 / NL;                           // load instructions per slot, operand and such a wavefront
  constexpr int CHUNK_UNITS = CHUNK_TILES * 32 / UNIT;
  static_assert((NW == 4 || NW == 8 || NLD == 4) && CHUNK_UNITS % NS == 0 && NS >= 2, "work-group shape");
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int b = blockIdx.y;
  // Work-groups are dealt to the eight XCDs round robin, each with an L2 of its own: with the KV head as the fastest
  // index every XCD serves the query blocks of the same few KV heads, and the keys those blocks share (every block
  // of a head walks the same keys) stay in ITS L2 instead of being fetched by all eight.
  // Causal attention: the last query blocks have the most keys, so they are dispatched first (longest work first
  // keeps the tail of the launch short); which work-group computes a block has no numeric effect.
  const int kvh = blockIdx.x % a.kv_heads;
  const int qb = gridDim.x / a.kv_heads - 1 - blockIdx.x / a.kv_heads;
  const int qlen = a.q_len[b];
  if (qb * ROWS >= qlen) return;  // uniform over the work-group
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ctx = a.ctx_len[b];
  // the tiles of 32 keys that the work-group's queries see; SPLIT: up to the end of chunk blockIdx.z
  const int tile0 = SPLIT ? (int)blockIdx.z * CHUNK_TILES : 0;
  const int all_tiles = (ctx - qlen + min(qb * ROWS + ROWS - 1, qlen - 1)) / 32 + 1;
  const int ntiles = SPLIT ? min(all_tiles, tile0 + CHUNK_TILES) : all_tiles;
  if (SPLIT && tile0 >= ntiles) return;  // uniform over the work-group
  const int unit0 = tile0 / 2, nunits = (ntiles + 1) / 2;

  // ---- staging: load instruction n of the sixteen of a slot covers key rows 4n .. 4n+3 / channel rows 8n .. 8n+7, 128 bytes of
  // each (whole lines of the V^T cache where its length is a multiple of 64); the wavefronts that load (all of them, or the NLD
  // loaders) deal them out in turn
  // A cache whose length is an odd number of tiles ends in the middle of the last slot: K instructions behind its end fetch
  // the last rows again, and V^T lanes of the second half what those of the first half do (rows that nobody sees).
  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.k_cache + ((int64_t)b * a.kv_heads + kvh) * a.max_len * HD);
  const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vt_cache + ((int64_t)b * a.kv_heads + kvh) * (int64_t)HD * a.max_len);
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int64_t vstep = (int64_t)a.max_len * 16;   // bytes of eight channel rows
  const int vchunk = (lane & 7) ^ v_swizzle(lane >> 3);
  const uint32_t vrow = (uint32_t)(lane >> 3) * (uint32_t)a.max_len * 2u;
  auto load_unit = [&](int unit, int slot) __attribute__((always_inline)) {
    const int k0 = min(unit * UNIT, a.max_len - 32);   // max_len is a multiple of 32
    const uint32_t voff = vrow + ((k0 + UNIT <= a.max_len ? vchunk : vchunk & 3) << 4);
#pragma unroll
    for (int i = 0; i < PI; i++) {
      const int n = (NLD ? wave - NW : wave) + i * NL;
      const int kr = 4 * n + (lane >> 4);
      const uint32_t koff = (uint32_t)((lane >> 4) * 256 + (((lane & 15) ^ k_swizzle(kr)) << 4));
      dma16(lds0 + slot * UNIT_BYTES + n * 1024, koff, kbase + (int64_t)min(k0 + 4 * n, a.max_len - 4) * (HD * 2));
      dma16(lds0 + slot * UNIT_BYTES + UNIT * HD * 2 + n * 1024, voff, vbase + (int64_t)k0 * 2 + n * vstep);
    }
  };

  // a slot has landed (this wavefront's share; up to NS - 2 slots stay in flight)
  auto landed = [&](int unit) __attribute__((always_inline)) { wait_slices<2 * PI, NS - 2>(min(NS - 2, nunits - 1 - unit)); };
  if (!NLD || wave >= NW) {
#pragma unroll
    for (int i = 0; i < NS - 1; i++)
      if (unit0 + i < nunits) load_unit(unit0 + i, i);
  }
  if (NLD && wave >= NW) {   // a loader: the barriers of the loop below, and nothing else of it
    for (int u0 = unit0; u0 < nunits; u0 += NS) {
#pragma unroll
      for (int d = 0; d < NS; d++) {
        const int unit = u0 + d;
        if (unit >= nunits) break;
        landed(unit);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (unit + NS - 1 < nunits) load_unit(unit + NS - 1, (d + NS - 1) % NS);
      }
    }
    return;
  }

  const int h = kvh * G + wave % G;
  const int j = lane & 15;
  const int g = lane >> 4;
  const int row0 = qb * ROWS + wave / G * (16 * QB);   // this wavefront's first query
  const int wave_tiles = min(ntiles, (ctx - qlen + min(row0 + 16 * QB - 1, qlen - 1)) / 32 + 1);
  int qpos[QB];
  bf16x8 qf[QB][4];
#pragma unroll
  for (int q = 0; q < QB; q++) {
    const int qrow = min(row0 + 16 * q + j, qlen - 1);
    qpos[q] = ctx - qlen + qrow;
    const uint16_t* qp = a.q + ((int64_t)(a.q_start[b] + qrow) * a.q_heads + h) * HD;
#pragma unroll
    for (int c = 0; c < 4; c++) qf[q][c] = *reinterpret_cast<const bf16x8*>(qp + c * 32 + g * 8);
  }

  f32x4 o[QB][8], ot[QB][8];   // this chunk's accumulators, and the merged chunks so far
  float m[QB], l[QB], mt[QB], lt[QB];
  auto empty_state = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < QB; q++) {
      m[q] = kNoKey, l[q] = 0.f;
#pragma unroll
      for (int t = 0; t < 8; t++) o[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  empty_state();
#pragma unroll
  for (int q = 0; q < QB; q++) mt[q] = lt[q] = 0.f;
  // chunk `c` is complete: merged into the rows that see it; after the last one the result stays in m, l and o,
  // otherwise an empty state follows
  auto end_chunk = [&](int c, bool last) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < QB; q++) {
      l[q] = row_sum(l[q]);
      if (c != 0) {
        if (qpos[q] >= c * CHUNK_TILES * 32) {
          float fa, fb;
          merge_chunk(mt[q], lt[q], m[q], l[q], fa, fb);
#pragma unroll
          for (int t = 0; t < 8; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) ot[q][t][i] = merge_acc(ot[q][t][i], fa, o[q][t][i], fb);
        }
      } else {
        mt[q] = m[q], lt[q] = l[q];
#pragma unroll
        for (int t = 0; t < 8; t++) ot[q][t] = o[q][t];
      }
      if (last) {
        l[q] = lt[q];
#pragma unroll
        for (int t = 0; t < 8; t++) o[q][t] = ot[q][t];
      }
    }
    if (!last) empty_state();
  };

  // fragment addresses in the first slot; every other slot, sub-tile and channel tile is an immediate offset from them
  typedef __attribute__((address_space(3))) const uint8_t lds_byte;
  typedef __attribute__((address_space(3))) const bf16x8 lds_fragment;
  lds_byte *kp[4], *vp[2];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    kp[c] = (lds_byte*)lds + k_fragment(j, c * 4 + g);
    asm volatile("" : "+v"(kp[c]));   // (the sum with the base of the LDS is formed once, not at every use)
  }
#pragma unroll
  for (int hf = 0; hf < 2; hf++) {
    vp[hf] = (lds_byte*)lds + UNIT * HD * 2 + v_fragment(j, hf * 4 + g);
    asm volatile("" : "+v"(vp[hf]));
  }
  // tile hf of the two in a slot.  All fragments of an operand are asked for before the first MFMA that takes one (the
  // scheduling barrier keeps the compiler from moving each read to its use, where the wave would wait out the LDS latency once
  // per fragment).
  auto read_keys = [&](int slot, int hf, bf16x8 (&kf)[4][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int u = 0; u < 2; u++) kf[c][u] = *(lds_fragment*)(kp[c] + slot * UNIT_BYTES + hf * 8192 + u * 1024);
  };
  auto read_values = [&](int slot, int hf, bf16x8 (&vf)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 8; t++) vf[t] = *(lds_fragment*)(vp[hf] + slot * UNIT_BYTES + t * 2048);
  };
  auto scores = [&](const bf16x8 (&kf)[4][2], int q, f32x4 (&s)[2]) __attribute__((always_inline)) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int u = 0; u < 2; u++) s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[c][u], qf[q][c], c == 0 ? zero : s[u], 0, 0, 0);
  };
  // mask and reference point of tile `tile`; the conditions are uniform over the wave
  auto reference = [&](int tile, int q, f32x4 (&s)[2]) __attribute__((always_inline)) {
    if (tile * 32 + 31 > ctx - qlen + row0 + 16 * q) mask_scores(s, tile * 32, g, qpos[q]);   // (beyond the block's first query)
    const float lmax = lane_max(s);
    if (__builtin_amdgcn_ballot_w64(score_exceeds(lmax, a.scale_log2, m[q])) != 0) {
      const float alpha = move_reference(lmax, a.scale_log2, m[q], l[q]);
#pragma unroll
      for (int t = 0; t < 8; t++) o[q][t] = f32x4{o[q][t][0] * alpha, o[q][t][1] * alpha, o[q][t][2] * alpha, o[q][t][3] * alpha};
    }
  };
  auto accumulate = [&](const bf16x8 (&vf)[8], int q, bf16x8 pf) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 8; t++) o[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t], pf, o[q][t], 0, 0, 0);
  };
  // eight MFMAs between the exponentials, so that neither kind comes in one long run: 1 - 3 % where a CU has one work-group (2 prompts of
  // 1020 tokens 31.3 -> 30.8 us, 1040 tokens of one head 16.6 -> 16.1, 526 at 3526 60.8 -> 59.9) or few rounds (prompts of 4096, 3136
  // and 2176 276 -> 271), level on the launches that fill the chip many times over
  auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);   // VALU
      __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);   // transcendental
    }
  };
  // formed here, and not behind the next branch where the compiler would sink it
  auto pin = [&](bf16x8& p, float& sum) __attribute__((always_inline)) {
    asm volatile("" : "+v"(p), "+v"(sum));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto do_tile = [&](int tile, int slot, int hf) __attribute__((always_inline)) {
    f32x4 s[QB][2];
    bf16x8 kf[4][2], vf[8], pf[QB];
    read_keys(slot, hf, kf);
    __builtin_amdgcn_sched_barrier(0);
    scores(kf, 0, s[0]);
    reference(tile, 0, s[0]);
#pragma unroll
    for (int q = 0; q < QB; q++) {
      if (q + 1 < QB) scores(kf, q + 1, s[q + 1]);
      else if (q > 0) accumulate(vf, q - 1, pf[q - 1]);
      if (q + 1 == QB - 1 || QB == 1) read_values(slot, hf, vf);
      pf[q] = probabilities(s[q], a.scale_log2, m[q], l[q]);
      interleave();
      pin(pf[q], l[q]);
      if (q + 1 < QB) reference(tile, q + 1, s[q + 1]);
    }
    accumulate(vf, QB - 1, pf[QB - 1]);
  };

  // The queries are in their registers from here on.  (The compiler does not see the direct loads: left to the first use, its
  // wait for the queries would stand in the loop and drain every load in flight.)
#pragma unroll
  for (int q = 0; q < QB; q++)
#pragma unroll
    for (int c = 0; c < 4; c++) asm volatile("" : "+v"(qf[q][c]));
  for (int c0 = unit0; c0 < nunits; c0 += CHUNK_UNITS) {
    const int ce = min(c0 + CHUNK_UNITS, nunits);
    for (int u0 = c0; u0 < ce; u0 += NS) {
#pragma unroll
      for (int d = 0; d < NS; d++) {   // slot d: a chunk is a whole number of rings
        const int unit = u0 + d;
        if (unit >= ce) break;
        // the slot has landed for every wave, and every wave is done with what it read from the slot before, which the
        // loads behind the barrier refill; up to NS - 2 slots stay in flight
        if (!NLD) landed(unit);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (!NLD && unit + NS - 1 < nunits) load_unit(unit + NS - 1, (d + NS - 1) % NS);
        if (2 * unit < wave_tiles) do_tile(2 * unit, d, 0);
        if (2 * unit + 1 < wave_tiles) do_tile(2 * unit + 1, d, 1);
      }
    }
    if (CHUNKS == ALL_CHUNKS && nunits > CHUNK_UNITS) end_chunk(c0 / CHUNK_UNITS, ce == nunits);
  }
  if (CHUNKS != ALL_CHUNKS || nunits <= CHUNK_UNITS) {
#pragma unroll
    for (int q = 0; q < QB; q++) l[q] = row_sum(l[q]);
  }
#pragma unroll
  for (int q = 0; q < QB; q++) {
    const int qrow = row0 + 16 * q + j;
    // (SPLIT: lengths are device data, and the workspace has rows for the caller's max_q_len, rounded up to 16)
    if (qrow >= qlen || (SPLIT && qrow >= sp.q_rows)) continue;
    if (SPLIT && qpos[q] >= 32 * CHUNK_TILES) {   // (a row that sees one chunk only is complete here)
      const int64_t at = ((int64_t)(b * sp.q_rows + qrow) * a.q_heads + h) * sp.nchunks + blockIdx.z;
#pragma unroll
      for (int t = 0; t < 8; t++) *reinterpret_cast<f32x4*>(sp.o + at * HD + 16 * t + 4 * g) = o[q][t];
      if (g == 0) *reinterpret_cast<f32x2*>(sp.ml + at * 2) = f32x2{m[q], l[q]};
      continue;
    }
    if (SPLIT && blockIdx.z != 0) continue;
    const float inv = 1.0f / l[q];
    uint16_t* op = a.out + ((int64_t)(a.q_start[b] + qrow) * a.q_heads + h) * HD;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const uint32_t lo = pack_bf16x2(o[q][t][0] * inv, o[q][t][1] * inv);
      const uint32_t hi = pack_bf16x2(o[q][t][2] * inv, o[q][t][3] * inv);
      *reinterpret_cast<uint2*>(op + 16 * t + 4 * g) = make_uint2(lo, hi);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Decode variant: every sequence brings so few new queries that all of them, for all G query heads of a KV head, fit
// the 16 rows of one MFMA tile (row = query * G + head of the group).  One work-group of eight wavefronts per
// (KV head, sequence):
//   * waves 0-3 compute.  All four form the scores and the softmax of the whole tile (the same instructions on the same
//     values, so the same bits in each) and each keeps the output accumulators of two of the eight 16-channel tiles: per
//     key tile a wave issues 8 + 2 MFMAs where a wave of the grouped kernel issues 16.  The scores of tile t + 1 are formed
//     before the softmax of tile t, so the MFMA chain of one tile runs beside the exponentials of the other.
//   * waves 4-7 do nothing but bring tiles in, with direct global->LDS loads (no staging registers, no LDS writes by a
//     wave): a decode step is one dependent chain of key tiles per sequence, and every load a computing wave issues is a
//     piece of that chain.  Loader i issues two of the eight 1 KiB load instructions of every K tile and four of the sixteen
//     of a pair of V^T tiles, 128 bytes of a channel row: whole lines of the value cache where the cache length is a
//     multiple of 64 (of an odd number of tiles, every second row begins in the middle of a line and its pieces touch two).
// The rows lie in LDS as k_swizzle and v_swizzle say.
// K tiles have a ring of NS slots, pairs of V^T tiles one of NP.  Iteration t reads K tile t + 1 and V^T tile t; the loaders request
// K tile t + NS (slot t % NS, read during iteration t - 1) and in every second iteration the pair of V^T tiles t + 2 NP - 2,
// t + 2 NP - 1 (the slot that iteration t - 1 finished), wait until what iteration t + 1 reads has landed (K tile t + 2, the
// pair of V^T tile t + 1; the counts follow from the order of the requests, and with the K ring's depth that order keeps a fourth
// slot of pairs from being any further ahead than a third), and all eight waves meet at the barrier.
// Only the first two K tiles and the first pair, 32 KB, are asked for without a look at the context (with two slots of pairs two more K
// tiles: 64 sequences of 300 keys 18.2 -> 17.8 us).  Requests behind its last tile ask for that one again (which
// comes from the L2; the tiles behind a context are up to 80 KB that nobody needs, a fifth of the
// traffic at 700 keys) and are never used, so the number of loads in flight is static; nothing is in flight when a wave ends.
// A row's arithmetic -- the lanes that own it, the MFMA chains over channels and key slots, the order of the softmax
// updates and of the chunks -- is that of the kernels above: the same bits.
// SPLIT: gridDim.z work-groups per (KV head, sequence); work-group z takes the chunks z, z + gridDim.z, ... as one stream of
// tiles and leaves each chunk's state in the workspace for attention_merge_kernel.  One work-group per (KV head,
// sequence) is a chain of 0.35 us per tile on as many CUs as there are such pairs: 8 sequences of 8000 keys 102 us before their
// chunks were spread over the chip (now 54, the merge included, in a cache of a multiple of 64 keys; the keys and values take 42
// at the rate of a one-pass read).
// ------------------------------------------------------------------------------------------------
template <int G, bool FUSED, bool SPLIT, int NP>
__global__ __launch_bounds__(512) void attention_decode_kernel(const AttnArgs a, const QkvArgs f, const SplitArgs sp) {
  constexpr int NS = 4;   // slots of K (tiles); NP of V^T (pairs of tiles)
  static_assert((NP == 2 || NP == 3) && CHUNK_TILES % NS == 0, "the waits below count these");
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_dyn[];
  uint8_t (*lds_k)[8192] = reinterpret_cast<uint8_t (*)[8192]>(lds_dyn);
  uint8_t (*lds_v)[16384] = reinterpret_cast<uint8_t (*)[16384]>(lds_dyn + NS * 8192);
  // FUSED: [G + 2][128] q heads, new key, new value, in the slot that the first iteration's loads refill
  uint16_t* hs = reinterpret_cast<uint16_t*>(lds_v[NP - 1]);
  constexpr int QMAX = 16 / G;
  constexpr int CT = 2;
  constexpr int NL = 4;               // loader waves
  constexpr int PI = 8 / NL;          // load instructions per loader wave and K tile; a pair of V^T tiles takes twice as many
  const int b = blockIdx.y;
  const int kvh = blockIdx.x;
  const int z = SPLIT ? blockIdx.z : 0, nz = SPLIT ? gridDim.z : 1;
  // tile i of this work-group's stream, and how many there are of ntiles in all
  auto tile_of = [&](int i) __attribute__((always_inline)) {
    return SPLIT ? (i / CHUNK_TILES * nz + z) * CHUNK_TILES + i % CHUNK_TILES : i;
  };
  auto tiles_here = [&](int ntiles) __attribute__((always_inline)) {
    if (!SPLIT) return ntiles;
    // lengths are device data: a sequence that ran off its cache has no chunk behind the last one of its slot in the
    // workspace, where the states of the next row begin (the merge is bounded likewise)
    ntiles = min(ntiles, a.max_len >> 5);
    const int nch = (ntiles + CHUNK_TILES - 1) / CHUNK_TILES;
    if (z >= nch) return 0;
    return (nch - z + nz - 1) / nz * CHUNK_TILES - ((nch - 1) % nz == z ? nch * CHUNK_TILES - ntiles : 0);
  };
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15;
  const int g = lane >> 4;
  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.k_cache + ((int64_t)b * a.kv_heads + kvh) * a.max_len * HD);
  const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vt_cache + ((int64_t)b * a.kv_heads + kvh) * (int64_t)HD * a.max_len);
  if (wv >= 4) {
    // ---------------- loader waves: loader li issues instructions li*PI .. li*PI+PI-1 of every K tile, 2*li*PI .. of a V^T pair
    const int li = wv - 4;
    // K: instruction q covers key rows 4q .. 4q+3 (1 KiB): lane -> row 4q + (lane >> 4), chunk position lane & 15
    // V^T: instruction q covers channel rows 8q .. 8q+7, 128 bytes each: lane -> row 8q + (lane >> 3), chunk position lane & 7
    // (a pair that reaches behind the cache: the second tile's lanes fetch what those of the first do, and nobody sees it)
    uint32_t kvoff[PI], vrow[2 * PI];
#pragma unroll
    for (int i = 0; i < PI; i++) {
      const int kr = 4 * (li * PI + i) + (lane >> 4), pc = lane & 15;
      kvoff[i] = (uint32_t)(kr * 256 + ((pc ^ k_swizzle(kr)) << 4));
    }
#pragma unroll
    for (int i = 0; i < 2 * PI; i++) vrow[i] = (uint32_t)(8 * (2 * li * PI + i) + (lane >> 3)) * (uint32_t)a.max_len * 2u;
    const int vchunk = (lane & 7) ^ v_swizzle(lane >> 3);   // (eight rows on, the swizzle is the same)
    const uint32_t lk = (uint32_t)(uintptr_t)&lds_k[0][0] + li * PI * 1024;
    const uint32_t lv = (uint32_t)(uintptr_t)&lds_v[0][0] + 2 * li * PI * 1024;
    auto load_k = [&](int tile, int slot) __attribute__((always_inline)) {
      const uint8_t* src = kbase + (int64_t)min(tile * 32, a.max_len - 32) * (HD * 2);
#pragma unroll
      for (int i = 0; i < PI; i++) dma16(lk + slot * 8192 + i * 1024, kvoff[i], src);
    };
    auto load_v = [&](int tile, int slot) __attribute__((always_inline)) {   // the pair that begins with tile `tile`
      const int k0 = min(tile * 32, a.max_len - 32);
      const uint8_t* src = vbase + (int64_t)k0 * 2;
      const uint32_t at = (uint32_t)((k0 + 64 <= a.max_len ? vchunk : vchunk & 3) << 4);
#pragma unroll
      for (int i = 0; i < 2 * PI; i++) dma16(lv + slot * 16384 + i * 1024, vrow[i] + at, src);
    };
    auto first_tiles = [&]() __attribute__((always_inline)) {
      load_k(tile_of(0), 0);
      load_k(tile_of(1), 1);
      load_v(tile_of(0), 0);
    };
    // on their way before the lengths are known, except where there may be no such chunk: in a cache that is mostly empty
    // most of these work-groups have nothing to do (8 sequences of 300 keys in a cache of 8192: 12.1 -> 9.0 us; the wait
    // costs full caches at most 1 us of 57)
    if (z == 0) first_tiles();
    if (NP == 2 && z == 0) {
      load_k(tile_of(2), 2);
      load_k(tile_of(3), 3);
    }
    const int ctx = a.ctx_len[b];
    const int qlen = FUSED ? (ctx > 0 ? 1 : 0) : a.q_len[b];
    if (qlen <= 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return;
    }
    const int last_pos = ctx - qlen + min(QMAX - 1, qlen - 1);
    const int ntiles = tiles_here(last_pos / 32 + 1);
    if (SPLIT && ntiles == 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return;
    }
    if (z != 0) first_tiles();
    const int last = max(ntiles - 1, 0);
    if (NP == 3 || z != 0) {
      load_k(tile_of(min(2, last)), 2);
      load_k(tile_of(min(3, last)), 3);
    }
    if (NP == 3) load_v(tile_of(min(2, last & ~1)), 1);
    if (FUSED) {
      // loaders 0 and 1 form the new key and file the new value while the first tiles are on their way (the computing
      // waves form the query heads meanwhile); everything they have in flight is drained before the barrier, so the waits
      // below still count the tile loads alone
      // (SPLIT: the work-group that has the position's chunk)
      if (li < 2 && (!SPLIT || ((ctx - 1) / (32 * CHUNK_TILES)) % nz == z)) {
        const int pos = ctx - 1;
        const uint16_t* src = f.qkv + (int64_t)b * f.ld + (int64_t)(a.q_heads + (li == 0 ? 0 : a.kv_heads) + kvh) * HD;
        const uint16_t r1 = src[lane], r2 = src[lane + 64];
        uint32_t o = (uint32_t)r1 | ((uint32_t)r2 << 16);
        if (li == 0) o = qk_norm_rope_head(r1, r2, f.kw, pos, f.inv_freq, f.eps, lane);
        hs[(G + li) * HD + lane] = (uint16_t)(o & 0xffffu);
        hs[(G + li) * HD + lane + 64] = (uint16_t)(o >> 16);
        if (pos < a.max_len) {
          if (li == 0) {
            uint16_t* dst = f.k_cache + (((int64_t)b * a.kv_heads + kvh) * a.max_len + pos) * HD;
            dst[lane] = (uint16_t)(o & 0xffffu);
            dst[lane + 64] = (uint16_t)(o >> 16);
          } else {
            uint16_t* dst = f.vt_cache + ((int64_t)b * a.kv_heads + kvh) * (int64_t)HD * a.max_len + pos;
            dst[(int64_t)lane * a.max_len] = r1;
            dst[(int64_t)(lane + 64) * a.max_len] = r2;
          }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      __syncthreads();  // the heads are in LDS
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * (NP == 2 ? 5 : 7)) : "memory");  // K tile 0
    __syncthreads();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * (NP == 2 ? 2 : 4)) : "memory");  // K tile 1, V^T pair 0
    __syncthreads();
    int vslot = NP - 1;   // of the pair that is asked for next
    for (int t0 = 0; t0 < ntiles; t0 += NS) {
#pragma unroll
      for (int d = 0; d < NS; d++) {
        const int tile = t0 + d;
        if (tile >= ntiles) break;
        load_k(tile_of(min(tile + NS, last)), d);   // slot of tile t, read during iteration t - 1
        if (d % 2 == 0) {
          load_v(tile_of(min(tile + 2 * NP - 2, last & ~1)), NP == 2 ? 1 - d / 2 : vslot);   // slot of the pair that iteration t - 1 finished
          vslot = vslot == NP - 1 ? 0 : vslot + 1;
        }
        // K tile t + 2, and the V^T pair of tile t + 1
        if (d % 2 == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * (NP == 2 ? 4 : 6)) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI * (NP == 2 ? 1 : 4)) : "memory");
        __syncthreads();
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  // ---------------- computing waves
  const int ctx = a.ctx_len[b];
  const int qlen = FUSED ? (ctx > 0 ? 1 : 0) : a.q_len[b];
  if (qlen <= 0) return;
  const int qi = j / G;
  const int h = kvh * G + j % G;
  const bool qvalid = qi < qlen;
  const int qrow = min(qi, qlen - 1);
  const int qpos = ctx - qlen + qrow;
  const int last_pos = ctx - qlen + min(QMAX - 1, qlen - 1);
  const int ntiles = tiles_here(last_pos / 32 + 1);
  if (SPLIT && ntiles == 0) return;
  const int nfull = (ctx - qlen + 1) / 32;
  bf16x8 qf[4];
  // FUSED: the G query heads of this (sequence, KV head) are formed here, one head per wave at a time, the key and the
  // value by two of the loader waves (per-head RMSNorm and rotary embedding as the stand-alone kernel does them); all are
  // left in LDS for the four computing waves and, the key and the value, filed in the caches for the steps to come.  This step takes them from LDS: the tile
  // that a loader brings in for their position holds whatever the cache held there, and is patched below.
  const int pos = ctx - 1;
  u32x4 new_k = {0, 0, 0, 0};   // lanes 0-15: the new key's chunk `lane`
  uint16_t new_v = 0;           // lanes 0-31: the new value's channel 32 wv + lane
  if (FUSED) {
    const uint16_t* row = f.qkv + (int64_t)b * f.ld;
    for (int u = wv; u < G; u += 4) {  // wave-uniform: the query heads (loaders 0 and 1 take the key and the value)
      const uint16_t* src = row + (int64_t)(kvh * G + u) * HD;
      const uint32_t o = qk_norm_rope_head(src[lane], src[lane + 64], f.qw, pos, f.inv_freq, f.eps, lane);
      hs[u * HD + lane] = (uint16_t)(o & 0xffffu);
      hs[u * HD + lane + 64] = (uint16_t)(o >> 16);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++) qf[c] = *reinterpret_cast<const bf16x8*>(hs + (j % G) * HD + c * 32 + g * 8);
    new_k = *reinterpret_cast<const u32x4*>(hs + G * HD + j * 8);
    new_v = hs[(G + 1) * HD + 16 * CT * wv + (lane & 31)];
  } else {
    const uint16_t* qp = a.q + ((int64_t)(a.q_start[b] + qrow) * a.q_heads + h) * HD;
#pragma unroll
    for (int c = 0; c < 4; c++) qf[c] = *reinterpret_cast<const bf16x8*>(qp + c * 32 + g * 8);
  }
  // the new key's row of the K tile in `slot` and the new value's column of this wave's rows of the V^T tile, from LDS
  // (each wave patches what it reads itself, right before it reads it: a wave's LDS operations keep their order)
  const int lt = pos >> 5, pr = pos & 31;
  auto patch_k = [&](int slot) __attribute__((always_inline)) {
    if (lane < 16)
      *reinterpret_cast<u32x4*>(&lds_k[slot][pr * 256 + ((lane ^ k_swizzle(pr)) << 4)]) = new_k;
  };
  auto patch_v = [&](int slot) __attribute__((always_inline)) {
    if (lane < 16 * CT) {
      const int ch = 16 * CT * wv + lane;
      *reinterpret_cast<uint16_t*>(&lds_v[slot][ch * 128 + (((4 * (lt & 1) + (pr >> 3)) ^ v_swizzle(ch)) << 4) + (pr & 7) * 2]) = new_v;
    }
  };
  uint32_t kofs[4];
#pragma unroll
  for (int c = 0; c < 4; c++) kofs[c] = k_fragment(j, c * 4 + g);
  uint32_t vofs[2];   // of the two tiles of a pair
#pragma unroll
  for (int hf = 0; hf < 2; hf++) vofs[hf] = CT * wv * 2048 + v_fragment(j, hf * 4 + g);
  auto scores = [&](int slot, f32x4 (&s)[2]) __attribute__((always_inline)) {
    const uint8_t* tb = &lds_k[slot][0];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      f32x4 acc;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(tb + kofs[c] + u * 1024);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[c], c == 0 ? zero : acc, 0, 0, 0);
      }
      s[u] = acc;
    }
  };
  f32x4 o[CT], ot[CT];
#pragma unroll
  for (int i = 0; i < CT; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNoKey, mt = 0.f;
  float l = 0.f, lsum = 0.f;
  __syncthreads();
  if (FUSED && tile_of(0) == lt) patch_k(0);
  f32x4 s_cur[2];
  scores(0, s_cur);
  __syncthreads();
  int vslot = 0;   // of this iteration's pair
  for (int c0 = 0; c0 < ntiles; c0 += CHUNK_TILES) {
    const int ce = min(c0 + CHUNK_TILES, ntiles);
    for (int t0 = c0; t0 < ce; t0 += NS) {
#pragma unroll
      for (int d = 0; d < NS; d++) {
        if (t0 + d >= ce) break;
        const int tile = tile_of(t0 + d), vs = NP == 2 ? d / 2 : vslot;
        if (FUSED && tile == lt) patch_v(vs);
        if (FUSED && tile_of(t0 + d + 1) == lt) patch_k((d + 1) % NS);
        bf16x8 vf[CT];
#pragma unroll
        for (int i = 0; i < CT; i++) vf[i] = *reinterpret_cast<const bf16x8*>(&lds_v[vs][vofs[d % 2] + i * 2048]);
        f32x4 s_next[2];
        scores((d + 1) % NS, s_next);
        if (tile >= nfull) mask_scores(s_cur, tile * 32, g, qpos);
        const float alpha = move_reference(lane_max(s_cur), a.scale_log2, m, l);
        const bf16x8 pf = probabilities(s_cur, a.scale_log2, m, l);
#pragma unroll
        for (int i = 0; i < CT; i++) o[i] = f32x4{o[i][0] * alpha, o[i][1] * alpha, o[i][2] * alpha, o[i][3] * alpha};
#pragma unroll
        for (int i = 0; i < CT; i++) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[i], pf, o[i], 0, 0, 0);
        __syncthreads();
        s_cur[0] = s_next[0];
        s_cur[1] = s_next[1];
        if (d % 2 == 1) vslot = vslot == NP - 1 ? 0 : vslot + 1;
      }
    }
    // the chunk is complete
    const int chunk = tile_of(c0) / CHUNK_TILES;
    l = row_sum(l);
    if (SPLIT && qpos >= 32 * CHUNK_TILES) {   // (a row that sees one chunk only is complete with it)
      if (qvalid) {
        const int64_t at = ((int64_t)(b * sp.q_rows + qi) * a.q_heads + h) * sp.nchunks + chunk;
#pragma unroll
        for (int i = 0; i < CT; i++) *reinterpret_cast<f32x4*>(sp.o + at * HD + 16 * (CT * wv + i) + 4 * g) = o[i];
        if (wv == 0 && g == 0) *reinterpret_cast<f32x2*>(sp.ml + at * 2) = f32x2{m, l};
      }
    } else if (chunk == 0) {
      mt = m, lsum = l;
#pragma unroll
      for (int i = 0; i < CT; i++) ot[i] = o[i];
    } else if (qpos >= chunk * CHUNK_TILES * 32) {
      float fa, fb;
      merge_chunk(mt, lsum, m, l, fa, fb);
#pragma unroll
      for (int i = 0; i < CT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) ot[i][e] = merge_acc(ot[i][e], fa, o[i][e], fb);
    }
    m = kNoKey, l = 0.f;
#pragma unroll
    for (int i = 0; i < CT; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (!qvalid || (SPLIT && (qpos >= 32 * CHUNK_TILES || z != 0))) return;
  const float inv = 1.0f / lsum;
  uint16_t* op = a.out + ((int64_t)(FUSED ? b : a.q_start[b] + qi) * a.q_heads + h) * HD + 16 * CT * wv;
#pragma unroll
  for (int i = 0; i < CT; i++) {
    const uint32_t lo = pack_bf16x2(ot[i][0] * inv, ot[i][1] * inv);
    const uint32_t hi = pack_bf16x2(ot[i][2] * inv, ot[i][3] * inv);
    *reinterpret_cast<uint2*>(op + 16 * i + 4 * g) = make_uint2(lo, hi);
  }
}

// The rows of several chunks, which different work-groups computed: one wavefront per (query, head), two channels per lane, the chunks
// merged in ascending order exactly as the kernels above merge them.  Sixteen chunks' loads are in flight at a time.
template <bool FUSED>
__global__ __launch_bounds__(256) void attention_merge_kernel(const AttnArgs a, const SplitArgs sp) {
  const int b = blockIdx.z, qi = blockIdx.y;
  const int h = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (h >= a.q_heads) return;
  // the lengths first: a row of one chunk is complete already, and of a cache that is mostly empty only the chunks in use
  // are read (states loaded while the lengths were on their way, all that the cache has room for, gained long contexts
  // nothing and cost short ones 1 .. 3 us)
  const int ctx = a.ctx_len[b];
  const int qlen = FUSED ? (ctx > 0 ? 1 : 0) : a.q_len[b];
  if (qi >= qlen) return;
  const int nch = min((ctx - qlen + qi) / (32 * CHUNK_TILES) + 1, sp.nchunks);
  if (nch <= 1) return;
  const int64_t at = ((int64_t)(b * sp.q_rows + qi) * a.q_heads + h) * sp.nchunks;
  const f32x2* po = reinterpret_cast<const f32x2*>(sp.o + at * HD) + lane;
  const f32x2* pm = reinterpret_cast<const f32x2*>(sp.ml + at * 2);
  constexpr int NB = 16;
  f32x2 O = {0.f, 0.f};
  float M = 0.f, L = 0.f;
  for (int c0 = 0; c0 < nch; c0 += NB) {
    f32x2 o[NB], ml[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int c = min(c0 + i, nch - 1);
      o[i] = po[(int64_t)c * (HD / 2)];
      ml[i] = pm[c];
    }
    if (c0 == 0) M = ml[0][0], L = ml[0][1], O = o[0];
#pragma unroll
    for (int i = 0; i < NB; i++) {
      if (c0 + i == 0) continue;
      if (c0 + i >= nch) break;
      float fa, fb;
      merge_chunk(M, L, ml[i][0], ml[i][1], fa, fb);
      O = f32x2{merge_acc(O[0], fa, o[i][0], fb), merge_acc(O[1], fa, o[i][1], fb)};
    }
  }
  const float inv = 1.0f / L;
  uint32_t* op = reinterpret_cast<uint32_t*>(a.out + ((int64_t)(FUSED ? b : a.q_start[b] + qi) * a.q_heads + h) * HD);
  op[lane] = pack_bf16x2(O[0] * inv, O[1] * inv);
}

static int chunks_of(int max_len) { return (max_len + 32 * CHUNK_TILES - 1) / (32 * CHUNK_TILES); }

// How many work-groups share the chunks of a (KV head, sequence) in the decode kernel: 1 = a single one walks them all.
// Enough for 512 work-groups in all, two per CU.  From 97 pairs on a chain per pair draws the keys nearly at the rate of
// the memory and the second launch is lost; with two chunks there is nothing to gain.  The lengths are the device's, so the
// rule has only the cache to go by: with few keys in a large cache the second launch is 2 us too many, from 1000 keys (64
// pairs) or 1500 (96) on the split wins (us, 8 KV heads, cache of 8192, one chain against split at 300, 600, 1000, 2000 and
// 8000 keys: 1 sequence 6.4 / 8.5, 9.9 / 12.1, 14.4 / 12.2, 25 / 12.3, 93 / 15; 8 sequences 6.6 / 9.0, 10.2 / 12.4,
// 16.0 / 13.0, 28 / 17, 102 / 57; 12 sequences 7.0 / 9.2, 10.8 / 14.3, 16.6 / 15.9, 29 / 27, 108 / 85; 16 sequences
// 7.3 / 12.5, 10.8 / 16.7, 15.5 / 20.0, 32 / 33, 122 / 120).
static int decode_split(int64_t pairs, int max_len) {
  const int nch = chunks_of(max_len);
  if (nch < 3 || pairs > 96) return 1;
  const int64_t want = 512 / pairs;
  return (int)(want > nch ? nch : want);
}
// The same for the grouped kernel, whose work-groups then take a chunk each: worth it while they are few (64 new tokens in
// a cache of 8192, one chain against split at 300, 600, 1000, 2000 and 8000 keys: 1 sequence 8.4 / 10.1, 13.1 / 15.9, 20 / 16,
// 36 / 17, 187 / 27; 4 sequences, 128 work-groups, 8.6 / 10.9, 13.8 / 22.4, 20 / 23, 44 / 30, 195 / 91).
static bool group_split(int64_t groups, int max_len) {
  const int nch = chunks_of(max_len);
  return nch >= 3 && groups <= 128 && groups * nch <= 2048;
}
static bool grouped_cache(int G, int kv_heads, int max_len) {
  return (max_len & 31) == 0 && (G == 1 || G == 2 || G == 4 || G == 8) && kv_heads <= 65535 && max_len <= (1 << 22);
}
// Queries per sequence that a call's tiles hold: all of a decode tile, or whole blocks of 16.
static int query_rows(int max_q_len, int G) { return (int64_t)max_q_len * G <= 16 ? 16 / G : (max_q_len + 15) / 16 * 16; }
size_t attention_workspace_bytes(int batch, int max_q_len, int q_heads, int kv_heads, int max_len) {
  if (batch <= 0 || max_q_len <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || max_len < 32) return 0;
  const int G = q_heads / kv_heads;
  if (!grouped_cache(G, kv_heads, max_len)) return 0;
  const bool split = (int64_t)max_q_len * G <= 16 ? decode_split((int64_t)batch * kv_heads, max_len) > 1
                                                  : group_split((int64_t)((max_q_len + 15) / 16) * kv_heads * batch, max_len);
  // A state is a row of 128 accumulators and two numbers.  The grouped kernel's bound above keeps them to 2^18 (130 MiB, at
  // 8 query heads per KV head); the decode kernel's is reached by 128 pairs with 65,536 keys each, which one work-group
  // per pair reads at the rate of the memory.
  const int64_t states = (int64_t)batch * query_rows(max_q_len, G) * q_heads * chunks_of(max_len);
  return split && states <= (1 << 18) ? (size_t)states * (HD + 2) * sizeof(float) : 0;
}
static SplitArgs split_args(void* ws, int batch, int max_q_len, int q_heads, int kv_heads, int max_len) {
  SplitArgs sp;
  sp.nchunks = chunks_of(max_len);
  sp.q_rows = query_rows(max_q_len, q_heads / kv_heads);
  sp.o = static_cast<float*>(ws);
  sp.ml = sp.o + (int64_t)batch * sp.q_rows * q_heads * sp.nchunks * HD;
  return sp;
}

template <bool FUSED>
static void merge_launch(const AttnArgs& a, const SplitArgs& sp, int batch, hipStream_t stream) {
  const dim3 grid((unsigned)((a.q_heads + 3) / 4), FUSED ? 1u : (unsigned)sp.q_rows, (unsigned)batch);
  hipLaunchKernelGGL(attention_merge_kernel<FUSED>, grid, dim3(256), 0, stream, a, sp);
}

template <int G, bool FUSED, bool SPLIT, int NP>
static int decode_run(const AttnArgs& a, const QkvArgs& f, const SplitArgs& sp, int batch, int nz, hipStream_t stream) {
  constexpr int LDS = 4 * 8192 + NP * 16384;
  static std::atomic<uint64_t> done{0};
  const hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(attention_decode_kernel<G, FUSED, SPLIT, NP>), LDS, done);
  if (e != hipSuccess) return hip_code(e);
  hipLaunchKernelGGL((attention_decode_kernel<G, FUSED, SPLIT, NP>), dim3((unsigned)a.kv_heads, (unsigned)batch, (unsigned)nz), dim3(512), LDS, stream, a, f, sp);
  return hip_code(hipGetLastError());
}

// Slots of V^T pairs: three (80 KiB of LDS with the K ring, two work-groups per CU), or two where all work-groups of a launch are
// resident at once and share the CUs: a deeper ring draws less from the memory there.  Measured on MI355X over 400 shapes (us,
// queries of one token, 4 heads over 8 unless stated; in parentheses with V^T tiles of 32 keys, half a line each, and tiles behind the context
// fetched; "same": contexts of one length, the others ragged), two slots / three:
//   up to 256 work-groups: 32 of 900 24.6 / 23.5 (24.8), 8 of 900 13.1 / 12.8 (14.5), 32 of 176 - / 7.5 (8.2), 30 of 106 7.4 / 6.5 (7.4);
//   257 .. 512: 8 of 8200 in a cache of 8224 59.5 / 65.6 (66.8), 48 of 1000 34.7 / 36.0 (41.0), 33 of 2707 78.3 / 82.6 (94.1),
//     40 of 3579 105.6 / 110.3 (122.4), 64 of 900 same 44.2 / 45.5 (44.5), 5 of 6870 34.0 / 33.3 (37.5), 12 of 8200 in 8224 92.0 / 93.5
//     (94.2), same 105.0 / 101.5 (100.5: the one shape found behind what it was);
//   more: 81 of 1397 87.2 / 79.3 (89.6), 128 of 1000 same 95.0 / 93.8 (91.4), 33 of 3723 of one head over 16 185.9 / 169.6 (177.8), 189 of
//     7508 same over 4 547.8 / 490.1 (490.4), 69 of 5195 of 8 heads same 312.7 / 285.5 (301.6), 112 of 151 of 8 heads 19.7 / 19.8 (26.7).
// Four slots are level with three up to 256 work-groups (the order of the requests again) and leave a CU room for one.
static bool two_pairs(int64_t wgs) { return wgs > 256 && wgs <= 512; }
template <int G, bool FUSED>
static int decode_launch(const AttnArgs& a, const QkvArgs& f, int batch, int max_q_len, void* ws, size_t ws_bytes, hipStream_t stream) {
  const int64_t pairs = (int64_t)batch * a.kv_heads;
  const size_t need = ws ? attention_workspace_bytes(batch, max_q_len, a.q_heads, a.kv_heads, a.max_len) : 0;
  if (need == 0 || ws_bytes < need)
    return two_pairs(pairs) ? decode_run<G, FUSED, false, 2>(a, f, SplitArgs{}, batch, 1, stream) : decode_run<G, FUSED, false, 3>(a, f, SplitArgs{}, batch, 1, stream);
  const SplitArgs sp = split_args(ws, batch, max_q_len, a.q_heads, a.kv_heads, a.max_len);
  const int nz = decode_split(pairs, a.max_len);
  const int rc = two_pairs(pairs * nz) ? decode_run<G, FUSED, true, 2>(a, f, sp, batch, nz, stream) : decode_run<G, FUSED, true, 3>(a, f, sp, batch, nz, stream);
  if (rc != TBIK_OK) return rc;
  merge_launch<FUSED>(a, sp, batch, stream);
  return hip_code(hipGetLastError());
}

template <int G, int WQ, int QB, int NS, int CHUNKS, int NLD>
static int group_run(const AttnArgs& a, const SplitArgs& sp, int batch, int max_q_len, hipStream_t stream) {
  constexpr int ROWS = 16 * QB * WQ, LDS = NS * UNIT_BYTES;
  const int64_t blocks = ((int64_t)max_q_len + ROWS - 1) / ROWS;
  const dim3 grid((unsigned)(blocks * a.kv_heads), (unsigned)batch, CHUNKS == SPLIT_CHUNKS ? (unsigned)sp.nchunks : 1u);
  static std::atomic<uint64_t> done{0};
  const hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(attention_group_kernel<G, WQ, QB, NS, CHUNKS, NLD>), LDS, done);
  if (e != hipSuccess) return hip_code(e);
  hipLaunchKernelGGL((attention_group_kernel<G, WQ, QB, NS, CHUNKS, NLD>), grid, dim3(64 * (G * WQ + NLD)), LDS, stream, a, sp);
  return hip_code(hipGetLastError());
}

// The form of the grouped kernel, same bits in all.  Lengths are the device's, so what is known is the number of
// work-groups, the queries of the longest sequence and the cache length -- its capacity, not the keys in it.
//   loaders: one block of 16 queries per wavefront and four more wavefronts that load, for launches of about one work-group per CU, which
//     are a chain of tiles (and up to several rounds where the cache is one chunk: without the merged chunks in registers two such
//     work-groups share a CU).  Two slots, and four (96 KiB of keys on their way) where keys were cached before: they come
//     from the memory, and the work-groups that share them ask at the same time.  Work-groups of one or two heads hold 64 or 32
//     queries, and 16 in a cache of one chunk while those are few: five or six wavefronts instead of eight.
//   plain: one block per wavefront, which loads for itself: two or three work-groups share a CU and fill each other's waits.
//   two blocks: per wavefront, half the fragment reads and half the key traffic per query, for launches that fill the chip in
//     twice as large pieces.  That takes more work-groups where the longest sequence is as long as the cache: with nothing
//     cached before it, its work-groups are of all lengths, and few large ones leave the chip with a tail.
//   Eight heads: plain only in one chunk (beside it another work-group fits a CU) and where work-groups take a chunk each (12 of 4 tokens
//     at 4511 keys 55 us, 64 with loaders); else loaders, and two blocks later than the others: a work-group of eight computing wavefronts
//     has twice the queries in flight already, and short or ragged sequences leave the second block empty.
// Measured on MI355X, us, loaders with two / with four slots, plain, two blocks (parentheses: the kernel with register staging and
// 16 queries per fragment read that these replace); the caches are as long as the longest context unless stated:
//   4 heads per KV head: 8192 tokens 724 / 769, 629, 503 (599), prompts of 4096, 3136 and 2176 358 / 396, 321, 256 (323), 1900 tokens
//     at 9000 keys 346 / 365, 297, 256 (299), 4 x 500 at 3000 130 / 137, 116, 100 (118), 32 x 64 at 4000 288 / 217, 195, 152 (182),
//     2 prompts of 1020 31 / 37, 29.3, 37 (41), 526 at 3526 71 / 75, 58, 73 (75), 1040 tokens 19.3 / 22.8, 21.4, 27.7 (26.9),
//     2 x 196 at 4251 50 / 51, 61, 88 (76), 4 x 128 at 8000 93 / 95, 113, 160 (138), 8 x 60 at 8000 118 / 97, 130, 161 (146),
//     24 x 16 at 4000 94 / 73, 94, 99 (80), one chunk: 16 x 400 45 / 66, 52, 47 (50), 32 x 512 144, -, 127;
//   the same in longer caches, where the rule takes them for cached keys: 2 prompts of 1020 in 8192 33.7 / 39.1, 31.8, 39.0 (42.7: two
//     blocks), 2000 tokens in 8192 56 / 61, 49.7, 50.7 (58.9: two blocks), 1040 tokens in 8192 -, 22.9 (28.2: plain), 16 x 400 in 4096
//     58 / 71, 56, 50.6 (53.4: two blocks);
//   8 heads: 4096 tokens 154 / 161, 165, 142 (185), 16 prompts of 400 in one chunk 49 / 54, 46, 55 (49), 32 x 64 at 4000 169 / 167, 176, 154
//     (208), 2 prompts of 1000 in 4096 28.4 / 28.9, 30.3, 38.6 (34.8), 36 x 37 at 3808 301 / 294, 309, 359 (311), 3 x 33 at 4649 46 / 45, 45,
//     57 (56), 38 x 10 at 6645 137 / 122, 139, 193 (159), 12 x 290 in 1216 51 / 53, 52, 55 (49), 4 x 4 5.5 / 5.6, 5.8, 6.3 (5.5);
//   2 heads: 8 x 400 at 4000 172 / 179, 147, 124 (184), 16 x 20 at 8000 151 / 102, 154, 165 (133), 300 at 2000 25.7 / 26.3, 30.0, 43 (34),
//     with 16 queries per work-group against 32: 4 x 38 4.9, 5.4 (5.1), 35 x 37 over 4 6.1, 7.7 (6.2), 61 x 19 over 4 7.1, 5.3 (7.6);
//   1 head: 4096 tokens 104 / 107, 91, 95 (133), 1040 tokens 15.1 / 16.0, 18.4, 24.5 (21.1), 16 queries per work-group against 64: 2 x 52
//     4.8, 5.4 (5.0);
//   with caches that hold nothing of it, 512 MB written in between: 2 x 196 at 4251 82 / 58, 88, 95 (84), 4 x 128 at 8000
//     139 / 103, 155, 168 (149), 300 at 2000 of 2 heads 42 / 30, 44, 49 (37), 526 at 3526 93 / 81, 73, 78 (83), 16 x 400 69 / 81, 71, 60 (66).
//   Over 919 random shapes (1 .. 64 sequences, 1 .. 8 heads over 1 .. 16, up to 4096 new tokens at up to 12,000 keys, caches of up to four times
//   that) the choice is 10 % ahead of the replaced kernel on average, and more than 5 % behind it (26 % at most) in one of 25: batches of
//   prompts of up to a few hundred tokens in caches of several chunks, where the registers of the merged chunks and slots of 64 keys keep
//   a third work-group from the CU.
//   (A load per wavefront that touches the lines of the unit behind the next costs a warm L2 5 - 25 % and was not kept.)
struct GroupForm {
  int wq, qb, ns, chunks, nld;   // the template arguments of group_run behind G
  bool operator==(const GroupForm& o) const { return wq == o.wq && qb == o.qb && ns == o.ns && chunks == o.chunks && nld == o.nld; }
};
static GroupForm group_form(int G, bool split, int batch, int max_q_len, int kv_heads, int max_len) {
  const int WQ = G >= 4 ? 1 : 4 / G;   // at least four computing wavefronts per work-group
  const int64_t blocks = ((int64_t)max_q_len + 15) / 16 * kv_heads * batch;
  const int64_t wgs = ((int64_t)max_q_len + 16 * WQ - 1) / (16 * WQ) * kv_heads * batch;
  const bool prompts = (int64_t)max_q_len * 4 > (int64_t)max_len * 3;
  if (split) return {WQ, 1, 2, SPLIT_CHUNKS, G == 8 ? 0 : 4};
  if (chunks_of(max_len) == 1) {
    if (blocks <= 256 || (wgs > 256 && blocks <= 512 && G < 4)) return {1, 1, 2, ONE_CHUNK, 4};
    if (G == 8) return {1, 1, 2, ONE_CHUNK, 0};
    if (max_q_len > 16 && wgs > 2500) return {WQ, 2, 2, ONE_CHUNK, 0};
    return {WQ, 1, 2, ONE_CHUNK, 4};
  }
  const bool two_blocks = G != 8 ? wgs > (prompts ? 1152 : 640)
                                 : wgs > 4500 || (max_q_len > 1200 && wgs > 1500) || (wgs > 850 && wgs > (int64_t)500 * batch);
  if (max_q_len > 16 && two_blocks) return {WQ, 2, 2, ALL_CHUNKS, 0};
  if (wgs <= 256 && (G == 8 ? max_q_len <= 64 && max_len >= 2048 : !prompts)) return {WQ, 1, 4, ALL_CHUNKS, 4};
  return {WQ, 1, 2, ALL_CHUNKS, G == 8 || (prompts && wgs <= 540) ? 4 : 0};
}
template <int G>
static int group_launch(const AttnArgs& a, const SplitArgs& sp, bool split, int batch, int max_q_len, hipStream_t stream) {
  constexpr int WQ = G >= 4 ? 1 : 4 / G;
  const GroupForm f = group_form(G, split, batch, max_q_len, a.kv_heads, a.max_len);
#define TBIK_ATTN_GROUP(...) if (f == GroupForm{__VA_ARGS__}) return group_run<G, __VA_ARGS__>(a, sp, batch, max_q_len, stream)
  TBIK_ATTN_GROUP(WQ, 1, 2, SPLIT_CHUNKS, G == 8 ? 0 : 4);
  TBIK_ATTN_GROUP(1, 1, 2, ONE_CHUNK, 4);
  TBIK_ATTN_GROUP(WQ, 1, 2, ALL_CHUNKS, 4);
  TBIK_ATTN_GROUP(WQ, 1, 4, ALL_CHUNKS, 4);
  TBIK_ATTN_GROUP(WQ, 2, 2, ALL_CHUNKS, 0);
  if constexpr (G == 8) {
    TBIK_ATTN_GROUP(1, 1, 2, ONE_CHUNK, 0);
  } else {
    if constexpr (WQ > 1) TBIK_ATTN_GROUP(WQ, 1, 2, ONE_CHUNK, 4);
    TBIK_ATTN_GROUP(WQ, 2, 2, ONE_CHUNK, 0);
    TBIK_ATTN_GROUP(WQ, 1, 2, ALL_CHUNKS, 0);
  }
#undef TBIK_ATTN_GROUP
  return TBIK_ERR_UNSUPPORTED;   // (a form that is not built)
}

// How a call would run (no effect on any result): out[0] kernel, 0 attention_kernel, 1 grouped, 2 decode; out[1] work-groups that
// share the chunks of a row; out[2] ring slots of 64 keys (1) or of V^T pairs (2); out[3] queries per work-group; out[4] blocks of 16
// queries per wavefront (1); out[5] wavefronts that load beside the computing ones (1, 2).
int attention_plan_info(int batch, int max_q_len, int q_heads, int kv_heads, int max_len, size_t ws_bytes, int out[6]) {
  if (!out || batch <= 0 || max_q_len <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || max_len < 32 || (max_len & 3)) return TBIK_ERR_INVALID;
  const int G = q_heads / kv_heads;
  const size_t need = attention_workspace_bytes(batch, max_q_len, q_heads, kv_heads, max_len);
  const bool split = need != 0 && ws_bytes >= need;
  for (int i = 0; i < 6; i++) out[i] = 0;
  out[1] = 1;
  if (!grouped_cache(G, kv_heads, max_len)) {
    out[3] = 16;
  } else if ((int64_t)max_q_len * G <= 16) {
    const int64_t pairs = (int64_t)batch * kv_heads;
    out[0] = 2;
    out[1] = split ? decode_split(pairs, max_len) : 1;
    out[2] = two_pairs(pairs * out[1]) ? 2 : 3;
    out[3] = 16 / G;
    out[5] = 4;
  } else {
    const GroupForm f = group_form(G, split, batch, max_q_len, kv_heads, max_len);
    out[0] = 1;
    out[1] = f.chunks == SPLIT_CHUNKS ? chunks_of(max_len) : 1;
    out[2] = f.ns;
    out[3] = 16 * f.wq * f.qb;
    out[4] = f.qb;
    out[5] = f.nld;
  }
  return TBIK_OK;
}

int attention_dispatch(const void* q, const void* k_cache, const void* vt_cache, void* out, const int* q_start,
                       const int* q_len, const int* ctx_len, int batch, int max_q_len, int q_heads, int kv_heads,
                       int head_dim, int max_len, float scale, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!q || !k_cache || !vt_cache || !out || !q_start || !q_len || !ctx_len) return TBIK_ERR_INVALID;
  if (batch <= 0 || max_q_len <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return TBIK_ERR_INVALID;
  if (head_dim != HD) return TBIK_ERR_UNSUPPORTED;
  if (max_len < 32 || (max_len & 3)) return TBIK_ERR_ALIGNMENT;
  auto mis = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
  if (mis(q) || mis(k_cache) || mis(vt_cache) || mis(out) || mis(ws)) return TBIK_ERR_ALIGNMENT;
  if (batch > 65535 || q_heads > 65535) return TBIK_ERR_INVALID;
  AttnArgs a{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k_cache), static_cast<const uint16_t*>(vt_cache),
             static_cast<uint16_t*>(out), q_start, q_len, ctx_len, q_heads, kv_heads, max_len, scale * 1.4426950408889634f};
  // the grouped kernel needs whole 32-key tiles in the caches, at most 8 query heads per KV head and a (sequence, head)
  // slice of a cache below 2 GiB (32-bit byte offsets)
  const int G = q_heads / kv_heads;
  const bool grouped = grouped_cache(G, kv_heads, max_len);
  if (grouped) {
    if ((int64_t)max_q_len * G <= 16) {  // all queries of a sequence and all heads of a group in one MFMA tile
      const QkvArgs none{};
      if (G == 1) return decode_launch<1, false>(a, none, batch, max_q_len, ws, ws_bytes, stream);
      if (G == 2) return decode_launch<2, false>(a, none, batch, max_q_len, ws, ws_bytes, stream);
      if (G == 4) return decode_launch<4, false>(a, none, batch, max_q_len, ws, ws_bytes, stream);
      return decode_launch<8, false>(a, none, batch, max_q_len, ws, ws_bytes, stream);
    }
    const int64_t gx = (int64_t)((max_q_len + 15) / 16) * kv_heads;
    if (gx > 0x7fffffff) return TBIK_ERR_INVALID;
    const size_t need = ws ? attention_workspace_bytes(batch, max_q_len, q_heads, kv_heads, max_len) : 0;
    const bool split = need != 0 && ws_bytes >= need;
    const SplitArgs sp = split ? split_args(ws, batch, max_q_len, q_heads, kv_heads, max_len) : SplitArgs{};
    const int code = G == 1 ? group_launch<1>(a, sp, split, batch, max_q_len, stream)
                   : G == 2 ? group_launch<2>(a, sp, split, batch, max_q_len, stream)
                   : G == 4 ? group_launch<4>(a, sp, split, batch, max_q_len, stream)
                            : group_launch<8>(a, sp, split, batch, max_q_len, stream);
    if (code != TBIK_OK) return code;
    if (split) merge_launch<false>(a, sp, batch, stream);
  } else {
    const dim3 grid((unsigned)((max_q_len + 15) / 16), (unsigned)q_heads, (unsigned)batch);
    hipLaunchKernelGGL(attention_kernel, grid, dim3(64), 0, stream, a);
  }
  return hip_code(hipGetLastError());
}

// One decode step of an attention block from the fused qkv projection output: per-head q/k RMSNorm, rotary embedding, the
// cache write and the attention of every sequence's one new token (row b of qkv, position ctx_len[b] - 1) in one launch.
// The bits of qk_norm_rope_cache_dispatch followed by attention_dispatch.  TBIK_ERR_UNSUPPORTED where the decode kernel
// does not apply (cache length not a whole number of tiles, more than 8 or an odd number of query heads per KV head):
// the caller makes the two calls.
int attention_decode_qkv_dispatch(const void* qkv, int64_t ld, const void* q_weight, const void* k_weight, const float* inv_freq,
                                  void* k_cache, void* vt_cache, void* out, const int* ctx_len, int batch, int q_heads,
                                  int kv_heads, int head_dim, int max_len, float scale, float eps, void* ws, size_t ws_bytes,
                                  hipStream_t stream) {
  if (!qkv || !q_weight || !k_weight || !inv_freq || !k_cache || !vt_cache || !out || !ctx_len) return TBIK_ERR_INVALID;
  if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return TBIK_ERR_INVALID;
  if (head_dim != HD) return TBIK_ERR_UNSUPPORTED;
  if (ld < (int64_t)(q_heads + 2 * kv_heads) * HD) return TBIK_ERR_INVALID;
  if (max_len < 32 || (max_len & 3)) return TBIK_ERR_ALIGNMENT;
  auto mis = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & m) != 0; };
  if (mis(k_cache, 15) || mis(vt_cache, 15) || mis(out, 15) || mis(ws, 15) || mis(qkv, 1) || mis(q_weight, 1) || mis(k_weight, 1) || mis(inv_freq, 3))
    return TBIK_ERR_ALIGNMENT;
  if (batch > 65535 || kv_heads > 65535) return TBIK_ERR_INVALID;
  const int G = q_heads / kv_heads;
  if ((max_len & 31) != 0 || !(G == 1 || G == 2 || G == 4 || G == 8) || max_len > (1 << 22)) return TBIK_ERR_UNSUPPORTED;
  AttnArgs a{nullptr, static_cast<const uint16_t*>(k_cache), static_cast<const uint16_t*>(vt_cache), static_cast<uint16_t*>(out),
             nullptr, nullptr, ctx_len, q_heads, kv_heads, max_len, scale * 1.4426950408889634f};
  const QkvArgs f{static_cast<const uint16_t*>(qkv), ld, static_cast<const uint16_t*>(q_weight), static_cast<const uint16_t*>(k_weight),
                  inv_freq, static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(vt_cache), eps};
  if (G == 1) return decode_launch<1, true>(a, f, batch, 1, ws, ws_bytes, stream);
  if (G == 2) return decode_launch<2, true>(a, f, batch, 1, ws, ws_bytes, stream);
  if (G == 4) return decode_launch<4, true>(a, f, batch, 1, ws, ws_bytes, stream);
  return decode_launch<8, true>(a, f, batch, 1, ws, ws_bytes, stream);
}

}  // namespace tbik
