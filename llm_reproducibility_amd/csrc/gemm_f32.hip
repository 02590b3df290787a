// fp32 GEMM for gfx950 with the same two accumulation disciplines as the 16-bit kernels:
//
//   TREE = true   tree-ordered (TP-invariant) matmul, the float32 branch of the reference's dtype-keyed
//                 configuration (leaf 128, src/tbik/tree_based_matmul.py:223-231): a leaf is the fp32 sum of its
//                 128 products, leaves merge through the binary counter (level 0 left to right over FLB leaves,
//                 adjacent pairs above), every node one fp32 addition.
//   TREE = false  one fp32 accumulator over all of K (aten::mm / aten::addmm on fp32 tensors in batch-invariant
//                 mode, src/bio/batch_invariant_ops.py:127-197).
//
// Products run on v_mfma_f32_16x16x4_f32 (full fp32 inputs; the reference's Triton dot uses TF32 on its hardware,
// so parity with it is to tolerance only).  K is walked in chunks of 16: a lane loads four consecutive k of its
// row (16 bytes) and the chunk's four MFMAs take k = 4g + j (g = lane / 16) -- a fixed permutation of the chunk,
// so the summation order of an element is a function of K alone: row m never sees M, tiles or the launch.
//
// Bound: the fp32 matrix rate (154 TFLOP/s in a large product on this card) from about 64 rows on, the weight stream below.
// A tile's operands go global -> LDS directly in slices of 32 k (128-byte rows, whole cache lines) through a ring of NS
// slots; fragments are read one chunk ahead of the MFMAs and the one barrier of a slice sits between its two chunks, so
// neither a memory round trip nor an LDS read is on the MFMA chain.  A wave's four MFMAs of an output tile and chunk are
// 128 cycles of matrix work per two 16-byte reads: neither the LDS nor the L2 is near its limit with any tile.  What is
// left is the barrier of a slice (a fifth of the time of a 64x64 tile); the tile is chosen for the grid (f32_pick).
#include "common.h"
#include "lds_direct.h"

namespace tbik {

struct GemmF32Args {
  const float* X;  // [M,K], row stride ldx
  const float* W;  // [N,K], row stride ldw
  float* C;        // [M,N], row stride ldc
  const float* bias;
  int64_t ldx, ldw, ldc;
  int M, N, K;
  int flb, lb;     // leaves of 128 per level-0 group, binary levels (TREE)
  int vec_store;
};

constexpr int F32_LBMAX = 8;
constexpr int F32_SLICE = 32;   // k per ring slot: 128 bytes per row

// WM x WN waves of TM x TN MFMA tiles (16x16) each; NS ring slots.
template <int WM, int WN, int TM, int TN, int NS>
struct F32Shape {
  static constexpr int NWAVE = WM * WN, RX = WM * TM * 16, RW = WN * TN * 16;
  static constexpr int NI = (RX + RW) / 8;      // direct loads (8 rows of 128 bytes each) per slice
  static constexpr int PI = NI / NWAVE;         // ... of which each wave issues
  static constexpr int STAGE = (RX + RW) * 128;
  static_assert(NI % NWAVE == 0 && NS >= 4 && PI * (NS - 2) < 64 && NS * STAGE <= 160 * 1024, "ring");
};

template <int WM, int WN, int TM, int TN, int NS, bool TREE>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_kernel(const GemmF32Args p) {
  typedef F32Shape<WM, WN, TM, TN, NS> S;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int tiles_m = (p.M + S::RX - 1) / S::RX;
  const int tiles_n = (p.N + S::RW - 1) / S::RW;
  // every XCD walks a contiguous range of tiles, eight rows of tiles at a time: neighbours share operand rows in its L2
  const int lid = xcd_contiguous_tile(blockIdx.x, gridDim.x);
  constexpr int GROUP = 8;
  const int first_m = (lid / (GROUP * tiles_n)) * GROUP;
  const int gsz = min(tiles_m - first_m, GROUP);
  const int in_group = lid % (GROUP * tiles_n);
  const int m0 = (first_m + in_group % gsz) * S::RX;
  const int n0 = (in_group / gsz) * S::RW;
  const int r16 = lane & 15, g = lane >> 4;

  const uint8_t* xbase = reinterpret_cast<const uint8_t*>(p.X + (int64_t)m0 * p.ldx);
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(p.W + (int64_t)n0 * p.ldw);
  // lane l of a load brings the 16-byte chunk that belongs at its linear place: row l / 8 of the eight, position l & 7,
  // where row r keeps chunk c at position c ^ (r & 7) (sixteen lanes of a fragment read then cover all banks)
  const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
  uint32_t voff[S::PI];
#pragma unroll
  for (int i = 0; i < S::PI; i++) {
    const int row = (wave * S::PI + i) * 8 + lrow;
    if (row < S::RX) voff[i] = (uint32_t)((int64_t)(min(m0 + row, p.M - 1) - m0) * p.ldx * 4) + lchunk * 16;
    else voff[i] = (uint32_t)((int64_t)(min(n0 + row - S::RX, p.N - 1) - n0) * p.ldw * 4) + lchunk * 16;
  }
  const int nchunks = p.K / 16;                // chunks of 16 k
  const int nslices = (nchunks + 1) / 2;
  // K may end in the middle of a slice: the lanes whose chunk lies behind it bring the first half again (never used)
  const uint32_t tail_back = (nchunks & 1) && lchunk >= 4 ? 64u : 0u;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  auto load_slice = [&](int s, int slot) __attribute__((always_inline)) {
    const int sc = min(s, nslices - 1);        // slices past the end load the last one again: the count in flight stays
    const uint32_t back = sc == nslices - 1 ? tail_back : 0u;
#pragma unroll
    for (int i = 0; i < S::PI; i++) {
      const int q = wave * S::PI + i;
      const uint8_t* b = (q < S::RX / 8 ? xbase : wbase) + (int64_t)sc * (F32_SLICE * 4);
      dma16(lds0 + slot * S::STAGE + q * 1024, voff[i] - back, b);
    }
  };
  const uint32_t frag = r16 * 128 + ((g ^ (r16 & 7)) << 4);
  const uint32_t xfrag = frag + wm * TM * 2048, wfrag = frag + S::RX * 128 + wn * TN * 2048;
  f32x4 fx[2][TM], fw[2][TN];
  auto read_frags = [&](int buf, int slot, int c) __attribute__((always_inline)) {
    const uint8_t* st = smem + slot * S::STAGE;
#pragma unroll
    for (int a = 0; a < TM; a++) fx[buf][a] = *reinterpret_cast<const f32x4*>(st + (xfrag ^ (c * 64)) + a * 2048);
#pragma unroll
    for (int b = 0; b < TN; b++) fw[buf][b] = *reinterpret_cast<const f32x4*>(st + (wfrag ^ (c * 64)) + b * 2048);
  };

  f32x4 acc[TM][TN];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) acc[a][b] = zero;
  auto multiply = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[buf][b][e], fx[buf][a][e], acc[a][b], 0, 0, 0);
  };

  // merge state (TREE): running level-0 sum and the binary counter's levels, all in registers
  constexpr int TA = TREE ? TM : 1, TB = TREE ? TN : 1;
  f32x4 s0[TA][TB], sb[TREE ? F32_LBMAX : 1][TA][TB];
  int c0 = 0, grp = 0;
  auto merge_leaf = [&](bool last) __attribute__((always_inline)) {
    // leaf done: binary-counter merge in fp32 (all conditions are uniform over the block)
    f32x4 t[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int b = 0; b < TB; b++) {
        t[a][b] = c0 != 0 ? s0[a][b] + acc[a][b] : acc[a][b];
        acc[a][b] = zero;
      }
    c0++;
    if (c0 == p.flb) {
      c0 = 0;
      bool parked = false;
#pragma unroll
      for (int l = 0; l < F32_LBMAX; l++) {
        if (!parked && l < p.lb) {
          if ((grp >> l) & 1) {
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
              for (int b = 0; b < TB; b++) t[a][b] = sb[l][a][b] + t[a][b];
          } else {
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
              for (int b = 0; b < TB; b++) sb[l][a][b] = t[a][b];
            parked = true;
          }
        }
      }
      grp++;
      if (last) {
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
          for (int b = 0; b < TB; b++) acc[a][b] = t[a][b];  // the root
      }
    } else {
#pragma unroll
      for (int a = 0; a < TA; a++)
#pragma unroll
        for (int b = 0; b < TB; b++) s0[a][b] = t[a][b];
    }
  };

  // prologue: NS - 1 slices in flight, slice 0 visible, its first fragments in registers
#pragma unroll
  for (int s = 0; s < NS - 1; s++) load_slice(s, s);
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(S::PI * (NS - 2)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_frags(0, 0, 0);
  int slot = 0;
  for (int s = 0; s < nslices; s++) {
    const int next = slot + 1 == NS ? 0 : slot + 1;
    const int prev = slot == 0 ? NS - 1 : slot - 1;
    read_frags(1, slot, 1);
    multiply(0);
    // slice s + 1 has landed (this wave's share) and every fragment read of slice s is done; behind the barrier the slot
    // of slice s - 1, which no wave reads any more, takes slice s + NS - 1
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(S::PI * (NS - 3)) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_slice(s + NS - 1, prev);
    read_frags(0, next, 0);
    if (2 * s + 1 < nchunks) multiply(1);
    if (TREE && (s & 3) == 3) merge_leaf(s == nslices - 1);   // a leaf of 128 is four slices
    slot = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // loads past the end of K have an address in this work-group's LDS

#pragma unroll
  for (int a = 0; a < TM; a++) {
    const int m = m0 + (wm * TM + a) * 16 + r16;
#pragma unroll
    for (int b = 0; b < TN; b++) {
      const int n = n0 + (wn * TN + b) * 16 + 4 * g;
      if (m >= p.M || n >= p.N) continue;
      float* dst = p.C + (int64_t)m * p.ldc + n;
      f32x4 v = acc[a][b];
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] += p.bias && n + e < p.N ? p.bias[n + e] : 0.f;
      if (p.vec_store && n + 3 < p.N) {
        *reinterpret_cast<f32x4*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < p.N) dst[e] = v[e];
      }
    }
  }
}

// The tree of few rows.  One chain over all of K is what a call of few rows waits for above, whatever the tile (31 us at K =
// 4096, 84 at 12288, where the weights need 11 and 32); a tree's leaves are independent, so here K is cut over the NW waves
// of a work-group of 16 columns, each an aligned subtree with a ring of its own in the LDS (no barrier until the end), and the
// waves' roots are added in adjacent pairs through the LDS: the same nodes, hence the same bits.  Rings of NS slices, so
// that eight waves are on a CU: one work-group of eight, or two of four; grid.y counts blocks of RX rows.
// [1,4096]x[4096,4096] 38.9 -> 13.3 us, [16,12288]x[12288,4096] 105 -> 41.5, [32,8192]x[8192,5120] 72 -> 61, [8,6144]x[6144,2048]
// 53 -> 15, weights from memory.  More rows as long as the blocks make at most two rounds ([64,6144]x[6144,2048] 54 -> 23,
// [128,6144]x[6144,2048] 55 -> 39, [64,4096]x[4096,4096] 38 -> 30, [64,12288]x[12288,4096] 106 -> 93); three rounds lose to the tiles.
template <int TM, int NW, int NS>
__global__ __launch_bounds__(64 * NW) void gemm_f32_strip_kernel(const GemmF32Args p) {
  constexpr int RX = TM * 16, STAGE = (RX + 16) * 128, NI = (RX + 16) / 8;
  static_assert(NS >= 3 && (NS - 1) * NI < 64 && NW * NS * STAGE <= 160 * 1024 && TM <= NW, "ring");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = xcd_contiguous_tile(blockIdx.x, gridDim.x) * 16, m0 = blockIdx.y * RX;
  const int r16 = lane & 15, g = lane >> 4;
  const int kw = p.K / NW, nslices = kw / F32_SLICE;  // this wave's k, a multiple of 128
  int lb = p.lb;
  for (int w = NW; w > 1; w >>= 1) lb--;
  const uint8_t* xbase = reinterpret_cast<const uint8_t*>(p.X + (int64_t)m0 * p.ldx + wave * kw);
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(p.W + (int64_t)n0 * p.ldw + wave * kw);
  const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
  uint32_t voff[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int row = i * 8 + lrow;  // X rows, then weight rows; rows past the edge are clamped
    if (row < RX) voff[i] = (uint32_t)((int64_t)(min(m0 + row, p.M - 1) - m0) * p.ldx * 4) + lchunk * 16;
    else voff[i] = (uint32_t)((int64_t)(min(n0 + row - RX, p.N - 1) - n0) * p.ldw * 4) + lchunk * 16;
  }
  uint8_t* ring = smem + wave * (NS * STAGE);
  const uint32_t lds0 = (uint32_t)(uintptr_t)ring;
  auto load_slice = [&](int s, int slot) __attribute__((always_inline)) {
    const int64_t at = (int64_t)min(s, nslices - 1) * (F32_SLICE * 4);  // past the end the last one again: the count in flight stays
#pragma unroll
    for (int i = 0; i < NI; i++) dma16(lds0 + slot * STAGE + i * 1024, voff[i], (i * 8 < RX ? xbase : wbase) + at);
  };
  const uint32_t frag = r16 * 128 + ((g ^ (r16 & 7)) << 4);
  f32x4 fx[2][2][TM], fw[2][2];
  auto read_frags = [&](int buf, int slot) __attribute__((always_inline)) {
    const uint8_t* st = ring + slot * STAGE;
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
      for (int a = 0; a < TM; a++) fx[buf][c][a] = *reinterpret_cast<const f32x4*>(st + (frag ^ (c * 64)) + a * 2048);
      fw[buf][c] = *reinterpret_cast<const f32x4*>(st + (frag ^ (c * 64)) + RX * 128);
    }
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TM], s0[TM], sb[F32_LBMAX][TM];
#pragma unroll
  for (int a = 0; a < TM; a++) acc[a] = zero;

#pragma unroll
  for (int s = 0; s < NS - 1; s++) load_slice(s, s);
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NS - 2) * NI) : "memory");
  read_frags(0, 0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  int slot = 0, c0 = 0, grp = 0;
  for (int j = 0; j < nslices / 4; j++) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int s = 4 * j + i, buf = i & 1;
      const int next = slot + 1 == NS ? 0 : slot + 1, prev = slot == 0 ? NS - 1 : slot - 1;
      // the slot of slice s - 1, whose fragments arrived a slice ago, takes slice s + NS - 1; then slice s + 1 has to be there
      load_slice(s + NS - 1, prev);
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NS - 2) * NI) : "memory");
      read_frags(buf ^ 1, next);
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int a = 0; a < TM; a++) acc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[buf][c][e], fx[buf][c][a][e], acc[a], 0, 0, 0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      slot = next;
    }
    // the leaf is done: binary-counter merge (all conditions are uniform)
    f32x4 t[TM];
#pragma unroll
    for (int a = 0; a < TM; a++) {
      t[a] = c0 != 0 ? s0[a] + acc[a] : acc[a];
      acc[a] = zero;
    }
    if (++c0 < p.flb) {
#pragma unroll
      for (int a = 0; a < TM; a++) s0[a] = t[a];
    } else {
      c0 = 0;
      bool parked = false;
#pragma unroll
      for (int l = 0; l < F32_LBMAX; l++) {
        if (!parked && l < lb) {
          if ((grp >> l) & 1) {
#pragma unroll
            for (int a = 0; a < TM; a++) t[a] = sb[l][a] + t[a];
          } else {
#pragma unroll
            for (int a = 0; a < TM; a++) sb[l][a] = t[a];
            parked = true;
          }
        }
      }
      grp++;
      if (!parked) {  // the wave's root, behind its last leaf
#pragma unroll
        for (int a = 0; a < TM; a++) s0[a] = t[a];
      }
    }
  }

  // roots of the waves, in the place of each wave's ring (its loads past the end of K have landed): adjacent pairs
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int a = 0; a < TM; a++) *reinterpret_cast<f32x4*>(ring + a * 1024 + lane * 16) = s0[a];
  __syncthreads();
  if (wave >= TM) return;  // wave a finishes tile a
  f32x4 v[NW];
#pragma unroll
  for (int w = 0; w < NW; w++) v[w] = *reinterpret_cast<const f32x4*>(smem + w * (NS * STAGE) + wave * 1024 + lane * 16);
#pragma unroll
  for (int d = 1; d < NW; d *= 2)
#pragma unroll
    for (int w = 0; w < NW; w += 2 * d) v[w] = v[w] + v[w + d];
  const int m = m0 + wave * 16 + r16, n = n0 + 4 * g;
  if (m >= p.M || n >= p.N) return;
  float* dst = p.C + (int64_t)m * p.ldc + n;
#pragma unroll
  for (int e = 0; e < 4; e++) v[0][e] += p.bias && n + e < p.N ? p.bias[n + e] : 0.f;
  if (p.vec_store && n + 3 < p.N) {
    *reinterpret_cast<f32x4*>(dst) = v[0];
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (n + e < p.N) dst[e] = v[0][e];
  }
}

template <int TM, int NW, int NS>
static int f32_strip_launch(const GemmF32Args& a, hipStream_t stream) {
  constexpr int smem = NW * NS * (TM * 16 + 16) * 128;
  auto kern = gemm_f32_strip_kernel<TM, NW, NS>;
  static std::atomic<uint64_t> done{0};
  hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, done);
  if (e != hipSuccess) return hip_code(e);
  hipLaunchKernelGGL(kern, dim3((unsigned)((a.N + 15) / 16), (unsigned)((a.M + TM * 16 - 1) / (TM * 16))), dim3(64 * NW), smem, stream, a);
  return hip_code(hipGetLastError());
}

// TBIK_ERR_UNSUPPORTED (nothing launched) where the tiles above serve the call
static int f32_strip(const GemmF32Args& a, hipStream_t stream) {
  const int64_t strips = ((int64_t)a.N + 15) / 16, blocks = ((int64_t)a.M + 31) / 32;
  if ((blocks > 1 && (strips * blocks > 512 || a.lb < 3)) || a.lb < 2 || a.ldx >= (1 << 24) || a.ldw >= (1 << 24)) return TBIK_ERR_UNSUPPORTED;  // 32-bit byte offsets
  const bool eight = a.lb >= 3 && strips <= 256;   // one round of work-groups of eight waves
  if (a.M <= 16) return eight ? f32_strip_launch<1, 8, 5>(a, stream) : f32_strip_launch<1, 4, 5>(a, stream);
  return eight ? f32_strip_launch<2, 8, 3>(a, stream) : f32_strip_launch<2, 4, 3>(a, stream);
}

template <int WM, int WN, int TM, int TN, int NS, bool TREE>
static int f32_launch(const GemmF32Args& a, hipStream_t stream) {
  typedef F32Shape<WM, WN, TM, TN, NS> S;
  const int64_t tiles = (int64_t)((a.M + S::RX - 1) / S::RX) * ((a.N + S::RW - 1) / S::RW);
  if (tiles > 0x7fffffff) return TBIK_ERR_INVALID;
  const int64_t reach = 0xffffff00ll - 128;   // byte offsets inside a tile's operand rows are 32 bits
  const int rx = a.M < S::RX ? a.M : S::RX, rw = a.N < S::RW ? a.N : S::RW;
  if ((rx > 1 && a.ldx > reach / 4 / (rx - 1)) || (rw > 1 && a.ldw > reach / 4 / (rw - 1))) return TBIK_ERR_UNSUPPORTED;
  static std::atomic<uint64_t> done{0};
  hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(gemm_f32_kernel<WM, WN, TM, TN, NS, TREE>), NS * S::STAGE, done);
  if (e != hipSuccess) return hip_code(e);
  hipLaunchKernelGGL((gemm_f32_kernel<WM, WN, TM, TN, NS, TREE>), dim3((unsigned)tiles), dim3(64 * S::NWAVE), NS * S::STAGE, stream, a);
  return hip_code(hipGetLastError());
}

// Which tile serves a call.  K cannot be cut (one accumulator, or one tree per element), so a call takes as many passes
// over K as the fullest CU has tiles, and the tile whose passes add up to the least time wins.  Microseconds of a pass at
// K = 4096 on MI355X, the first (launch and first loads included, 256 tiles) and each further one:
//   mm    32x32, 4 waves 32 / 23.5   64x32, 4 waves 46.5 / 36.5   64x64, 16 waves 83 / 66.5   128x128, 8 waves 247 / 249
//   tree  32x32, 4 waves 40 / 26     64x64, 16 waves 84 / 81
// (matrix work alone: 13.7, 27.3, 54.6 and 218 us).  Several small waves per SIMD beat few large ones: 64x64 with four
// waves of 32x32 takes 78 us for mm and 111 for the tree, whose merges then stand in the MFMAs' way.  Whole calls, before
// (operands read straight from global memory, nothing prefetched) -> after: mm [256,4096]x[4096,4096] 136 -> 78 us,
// [2048,4096]x[4096,6144] 1519 -> 745 (138 TFLOP/s), [16,4096]x[4096,4096] 114 -> 30; tree 139 -> 84, 1390 -> 969, 118 -> 38.
struct F32Tile {
  int rows, cols;
  double first, next;
};
static int f32_pick(int M, int N, int K, bool tree) {
  static const F32Tile mm[4] = {{32, 32, 32., 23.5}, {64, 32, 46.5, 36.5}, {64, 64, 83., 66.5}, {128, 128, 247., 249.}};
  static const F32Tile tr[4] = {{32, 32, 40., 26.}, {64, 32, 1e9, 1e9}, {64, 64, 84., 81.}, {128, 128, 1e9, 1e9}};
  int best = 0;
  double best_t = 0.;
  for (int c = 0; c < 4; c++) {
    const F32Tile& t = tree ? tr[c] : mm[c];
    const int64_t tiles = (((int64_t)M + t.rows - 1) / t.rows) * (((int64_t)N + t.cols - 1) / t.cols);
    const double k = K / 4096.0;
    const double us = 5.0 + (t.first - 5.0) * k + t.next * k * (double)((tiles + 255) / 256 - 1);
    if (c == 0 || us < best_t) {
      best_t = us;
      best = c;
    }
  }
  return best;
}

template <bool TREE>
static int f32_run(const GemmF32Args& a, int cfg, hipStream_t stream) {
  if (cfg == 0) return f32_launch<2, 2, 1, 1, 8, TREE>(a, stream);
  if (cfg == 2 || TREE) return f32_launch<4, 4, 1, 1, 4, TREE>(a, stream);
  if (cfg == 1) return f32_launch<2, 2, 2, 1, 6, false>(a, stream);
  return f32_launch<2, 4, 4, 2, 4, false>(a, stream);
}

// Rows so far apart that a tile's rows do not fit 32-bit offsets (138 MB for 32 rows) go to the smallest tile, which reaches
// furthest, and beyond that to halves of the product: a single row has no distance to the next.
template <bool TREE>
static int f32_run_reaching(const GemmF32Args& a, int cfg, hipStream_t stream) {
  int rc = f32_run<TREE>(a, cfg, stream);
  if (rc == TBIK_ERR_UNSUPPORTED && cfg != 0) rc = f32_run<TREE>(a, 0, stream);
  if (rc != TBIK_ERR_UNSUPPORTED || (a.M == 1 && a.N == 1)) return rc;
  GemmF32Args lo = a, hi = a;
  if (a.N == 1 || (a.M > 1 && a.ldx >= a.ldw)) {
    lo.M = a.M / 2;
    hi.M = a.M - lo.M;
    hi.X += (int64_t)lo.M * a.ldx;
    hi.C += (int64_t)lo.M * a.ldc;
  } else {
    lo.N = a.N / 2;
    hi.N = a.N - lo.N;
    hi.W += (int64_t)lo.N * a.ldw;
    hi.C += lo.N;
    if (a.bias) hi.bias += lo.N;
    hi.vec_store = a.vec_store && (lo.N & 3) == 0;
  }
  rc = f32_run_reaching<TREE>(lo, 0, stream);
  return rc == TBIK_OK ? f32_run_reaching<TREE>(hi, 0, stream) : rc;
}

int gemm_f32_dispatch(bool tree, const void* A, int64_t lda, const void* B, int64_t ldb_k, int64_t ldb_n, void* C,
                      int64_t ldc, int M, int N, int K, int leaf_k, const void* bias, hipStream_t stream) {
  if (M < 0 || N < 0 || K <= 0) return TBIK_ERR_INVALID;
  if (M == 0 || N == 0) return TBIK_OK;
  if (!A || !B || !C) return TBIK_ERR_INVALID;
  if (ldb_k != 1) return TBIK_ERR_UNSUPPORTED;  // row-major [K,N] weights are repacked by the caller
  if (lda < K || ldb_n < K || ldc < N) return TBIK_ERR_INVALID;
  auto mis = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) != 0; };
  if (mis(A) || mis(B) || (lda & 3) || (ldb_n & 3) || (K & 15)) return TBIK_ERR_ALIGNMENT;
  if (reinterpret_cast<uintptr_t>(C) & 3) return TBIK_ERR_ALIGNMENT;
  GemmF32Args a{static_cast<const float*>(A), static_cast<const float*>(B), static_cast<float*>(C),
                static_cast<const float*>(bias), lda, ldb_n, ldc, M, N, K, 1, 0, (ldc & 3) == 0 && !mis(C)};
  if (tree) {
    if (leaf_k != 128) return TBIK_ERR_UNSUPPORTED;
    int T, flb, level_k;
    if (tbik_tree_params(K, leaf_k, &T, &flb, &level_k) != TBIK_OK) return TBIK_ERR_INVALID;
    if (level_k - 1 > F32_LBMAX) return TBIK_ERR_UNSUPPORTED;
    a.flb = flb;
    a.lb = level_k - 1;
    const int rc = f32_strip(a, stream);
    if (rc != TBIK_ERR_UNSUPPORTED) return rc;
  }
  const int cfg = f32_pick(M, N, K, tree);
  return tree ? f32_run_reaching<true>(a, cfg, stream) : f32_run_reaching<false>(a, cfg, stream);
}

}  // namespace tbik
