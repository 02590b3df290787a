// Tree-ordered 16-bit GEMM for gfx950, decode batches (up to 64 rows): one pass over the weights through a deep LDS ring.
// Replaces matmul_kernel_tp_persistent, src/tbik/tree_based_matmul.py:50-187, at the row counts where the weights are
// nearly all of the traffic.
//
// What bounds it: bytes in flight.  256 CUs share 6.2 TB/s at well over a microsecond of latency, so a CU has to keep
// some 50 KB asked for.  The tiled kernel (gemm_tiled.hip) stages through registers two slices of 16 KiB ahead and ran at
// 4.0 - 4.6 TB/s here; a ring of direct global->LDS loads costs no registers and takes all the LDS there is.
//
// A work-group is NW waves of 32 columns each over all rows (MT tiles of 16); a slice is 64 of K.  Wave w loads the
// weight rows that it alone multiplies and its share of the X rows, NSLOT - 1 slices ahead; one barrier per slice.  NW is
// chosen so that the tiles times the K split put the same number of work-groups on every CU (5120 columns are 32 tiles
// of 160, eight K shards: 256 work-groups; tiles of 128 would be 320).
//
// Measured with cold weights, shard combine included, tiled kernel -> this: [49,25600]x[25600,5120] 67.1 -> 56.9 us,
// [32,25600]x[25600,5120] 63.3 -> 53.0 (5.0 TB/s), [32,8192]x[8192,5120] 25.0 -> 20.2, [32,12288]x[12288,4096] 25.9 -> 24.3,
// [16,12288]x[12288,4096] 24.2 -> 23.2; never behind by more than 2 % over 5 .. 64 rows of nine layer shapes.  Over 1479 points
// of N = 64 .. 51200 and K = 256 .. 32768 8 % faster on average, 8 % of them more than 4 % slower: a few rows on tiny
// matrices (0.4 .. 1 us) and N = 16384 and more on a K cut in two ([32,12288]x[12288,16384] 80 -> 97).
//
// Weights of 64 MB and more are loaded with the non-temporal hint (dma16_once) up to 32 rows, as a model's are in decode: from
// memory on every call.  Without it -> with it, us, weights from memory / the same ones again and again / copied into place just before:
//   [16,25600]x[25600,5120] 52.9 -> 47.4 / 44.1 -> 46.2 / 54.2 -> 59.8;  [16,12288]x[12288,4096] 24.1 -> 21.9 / 20.4 -> 20.0 / 22.4 -> 22.1;
//   [32,12288]x[12288,4096] 25.1 -> 22.9 / 21.6 -> 21.3 / 24.0 -> 23.8;  [32,8192]x[8192,5120] 20.7 -> 19.6 / 18.7 -> 18.2 / 21.0 -> 20.5.
// It is off where it gives little from memory or takes more from weights that the 256 MB cache holds: smaller ones ([8,4096]x[4096,4096]
// 11.3 -> 10.9 / 8.4 -> 8.7 / 13.4 -> 13.3) and more rows ([49,25600]x[25600,5120] 58.7 -> 58.3 / 55.9 -> 56.4 / 66.2 -> 64.5, written in place
// just before 64.0 -> 72.7; [64,8192]x[8192,5120] 25.4 -> 25.6 / 22.0 -> 21.9 / 24.5 -> 31.6; [49,12288]x[12288,4096] 26.5 -> 24.5 / 23.2 ->
// 23.1 / 25.5 -> 30.8).
//
// The arithmetic per element is that of gemm_tiled.hip: one chain of 16x16x32 MFMAs over ascending k per leaf, one
// rounding per leaf, left to right over the leaves of a group, adjacent pairs above, every node rounded; the whole tree
// of a shard lives in registers.  Hence the same bits.
#include <type_traits>

#include "common.h"
#include "gemm_args.h"
#include "lds_direct.h"

namespace tbik {

namespace few {
constexpr int BK = 64, TN = 2;
constexpr int LBMAX = TREE_FEW_LEVELS;  // more would not fit the registers of five or six waves
template <int MT, int NW>
struct Shape {
  static constexpr int BN = NW * TN * 16;
  static constexpr int STAGE_BYTES = (MT * 16 + BN) * BK * 2;
  static constexpr int XDMA = (MT * 2 + NW - 1) / NW;  // direct loads of 8 X rows per wave and slice
  static constexpr int WDMA = TN * 2;                  // ... of 8 weight rows: the wave's own 32
  static constexpr int NDMA = XDMA + WDMA;
  // all of the LDS, as far as the counter of outstanding loads (63) and a short shard (8 slices) make use of it
  static constexpr int FIT = 160 * 1024 / STAGE_BYTES;
  static constexpr int CNT = 63 / NDMA + 1;
  static constexpr int NSLOT = FIT < CNT ? (FIT < 8 ? FIT : 8) : (CNT < 8 ? CNT : 8);
};
}  // namespace few

// MT: 16-row tiles; NW: waves, 32 columns each; LS: slices per leaf; ONCE: weights with the non-temporal hint
template <int MT, int NW, int LS, bool F16, bool ONCE>
__global__ __launch_bounds__(NW * 64) void gemm_tree_few_kernel(const WideArgs p) {
  using namespace few;
  using Num = Num16<F16>;
  using S = Shape<MT, NW>;
  constexpr int NSLOT = S::NSLOT, NDMA = S::NDMA, XDMA = S::XDMA, NREG = MT * TN * 2;
  static_assert(NSLOT >= 3, "ring");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int shard = blockIdx.y;
  const int n0 = xcd_contiguous_tile(blockIdx.x, gridDim.x) * S::BN;

  const uint8_t* xbase = reinterpret_cast<const uint8_t*>(p.X + shard * p.k_shard);
  const uint8_t* wbase = reinterpret_cast<const uint8_t*>(p.W + (int64_t)n0 * p.ldw + shard * p.k_shard);
  // byte offsets of this lane's loads and the LDS place of each; rows past the edge are clamped (their results are not
  // stored).  Where NW does not divide the X rows the last waves load the last group once more: same bytes, same place.
  uint32_t voff[NDMA], dst[NDMA];
  {
    const int r = lane >> 3, c = (lane & 7) ^ r;
#pragma unroll
    for (int i = 0; i < XDMA; i++) {
      const int grp = min(i * NW + wave, 2 * MT - 1);
      voff[i] = (uint32_t)(((int64_t)min(grp * 8 + r, p.M - 1) * p.ldx + c * 8) * 2);
      dst[i] = grp * 1024;
    }
#pragma unroll
    for (int i = 0; i < S::WDMA; i++) {
      const int row = wave * TN * 16 + i * 8;
      voff[XDMA + i] = (uint32_t)(((int64_t)(min(n0 + row + r, p.N - 1) - n0) * p.ldw + c * 8) * 2);
      dst[XDMA + i] = (MT * 16 + row) * 128;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  auto issue = [&](int s, int slot) __attribute__((always_inline)) {
    const uint32_t base = lds0 + slot * S::STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < XDMA; i++) dma16(base + dst[i], voff[i], xbase + (int64_t)s * (BK * 2));
#pragma unroll
    for (int i = XDMA; i < NDMA; i++) {
      if (ONCE) dma16_once(base + dst[i], voff[i], wbase + (int64_t)s * (BK * 2));
      else dma16(base + dst[i], voff[i], wbase + (int64_t)s * (BK * 2));
    }
  };

  const int frow = lane & 15, fchk = lane >> 4;
  const uint32_t xfrag = (frow * BK + ((fchk ^ (frow & 7)) << 3)) * 2;
  const uint32_t wfrag = ((MT * 16 + wave * TN * 16 + frow) * BK + ((fchk ^ (frow & 7)) << 3)) * 2;

  f32x4 acc[MT][TN];
  uint32_t t[NREG], s0[NREG], sb[LBMAX][NREG];
#pragma unroll
  for (int r = 0; r < NREG; r++) {
    t[r] = s0[r] = 0;
#pragma unroll
    for (int l = 0; l < LBMAX; l++) sb[l][r] = 0;
  }

  const int nst = p.T * LS;
#pragma unroll
  for (int s = 0; s < NSLOT - 1; s++)
    if (s < nst) issue(s, s);

  int slot = 0, pos = 0, g = 0, s = 0;
  for (int j = 0; j < p.T; j++) {
#pragma unroll
    for (int i = 0; i < LS; i++, s++) {
      wait_slices<NDMA, NSLOT - 2>(nst - 1 - s);         // slice s has landed, this wave's share of it
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave has read slice s - 1
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (s + NSLOT - 1 < nst) issue(s + NSLOT - 1, slot == 0 ? NSLOT - 1 : slot - 1);  // over slice s - 1
      const uint8_t* base = smem + slot * S::STAGE_BYTES;
      bf16x8 fx[2][MT], fw[2][TN];
#pragma unroll
      for (int kk = 0; kk < 2; kk++) {
#pragma unroll
        for (int b = 0; b < TN; b++) fw[kk][b] = *reinterpret_cast<const bf16x8*>(base + (wfrag ^ (kk * 64)) + b * 16 * BK * 2);
#pragma unroll
        for (int a = 0; a < MT; a++) fx[kk][a] = *reinterpret_cast<const bf16x8*>(base + (xfrag ^ (kk * 64)) + a * 16 * BK * 2);
      }
#pragma unroll
      for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
          for (int b = 0; b < TN; b++) {
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            acc[a][b] = Num::mfma(fw[kk][b], fx[kk][a], (i == 0 && kk == 0) ? zero : acc[a][b]);
          }
      slot = slot + 1 == NSLOT ? 0 : slot + 1;
    }
    // the finished leaf: into the running sum of its group, a finished group up the binary levels
#pragma unroll
    for (int a = 0; a < MT; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) {
        t[(a * TN + b) * 2] = Num::pack(acc[a][b][0], acc[a][b][1]);
        t[(a * TN + b) * 2 + 1] = Num::pack(acc[a][b][2], acc[a][b][3]);
      }
    if (pos != 0) {
#pragma unroll
      for (int r = 0; r < NREG; r++) t[r] = Num::add(s0[r], t[r]);
    }
    if (pos + 1 < p.flb) {
#pragma unroll
      for (int r = 0; r < NREG; r++) s0[r] = t[r];
      pos++;
    } else {
      pos = 0;
      bool carry = true;
#pragma unroll
      for (int l = 0; l < LBMAX; l++) {
        if (carry && l < p.lb) {
          if ((g >> l) & 1) {
#pragma unroll
            for (int r = 0; r < NREG; r++) t[r] = Num::add(sb[l][r], t[r]);
          } else {
#pragma unroll
            for (int r = 0; r < NREG; r++) sb[l][r] = t[r];
            carry = false;
          }
        }
      }
      g++;
    }
  }

#pragma unroll
  for (int a = 0; a < MT; a++) {
    const int m = a * 16 + frow;
#pragma unroll
    for (int b = 0; b < TN; b++) {
      const int n = n0 + (wave * TN + b) * 16 + fchk * 4;
      if (m >= p.M || n >= p.N) continue;
      uint32_t lo = t[(a * TN + b) * 2], hi = t[(a * TN + b) * 2 + 1];
      if (p.bias) {
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < p.N) bv[e] = Num::to_f32(p.bias[n + e]);
        lo = Num::add(lo, Num::pack(bv[0], bv[1]));
        hi = Num::add(hi, Num::pack(bv[2], bv[3]));
      }
      uint16_t* out = p.C + shard * p.c_shard + (int64_t)m * p.ldc + n;
      if (p.vec_store && n + 3 < p.N) {
        *reinterpret_cast<uint2*>(out) = make_uint2(lo, hi);
      } else {
        const uint16_t v[4] = {(uint16_t)(lo & 0xffff), (uint16_t)(lo >> 16), (uint16_t)(hi & 0xffff), (uint16_t)(hi >> 16)};
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < p.N) out[e] = v[e];
      }
    }
  }
}

template <int MT, int NW, int LS, bool F16, bool ONCE>
static int few_launch(const WideArgs& a, int split, hipStream_t stream) {
  using namespace few;
  using S = Shape<MT, NW>;
  constexpr int smem = S::NSLOT * S::STAGE_BYTES;
  static_assert(smem <= 160 * 1024 && (S::NSLOT - 1) * S::NDMA < 64, "ring does not fit the LDS or the wait counter");
  static std::atomic<uint64_t> done{0};
  hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(gemm_tree_few_kernel<MT, NW, LS, F16, ONCE>), smem, done);
  if (e != hipSuccess) return hip_code(e);
  const unsigned tiles = (unsigned)((a.N + S::BN - 1) / S::BN);
  hipLaunchKernelGGL((gemm_tree_few_kernel<MT, NW, LS, F16, ONCE>), dim3(tiles, (unsigned)split), dim3(NW * 64), smem, stream, a);
  return hip_code(hipGetLastError());
}

template <int LS, bool F16>
static int few_by_shape(const WideArgs& a, int waves, int split, hipStream_t stream) {
  const bool once = (int64_t)a.N * a.K * split * 2 >= 64000000;
  auto rows = [&](auto nw) {
    constexpr int NW = decltype(nw)::value;
    if (a.M <= 16) return once ? few_launch<1, NW, LS, F16, true>(a, split, stream) : few_launch<1, NW, LS, F16, false>(a, split, stream);
    if (a.M <= 32) return once ? few_launch<2, NW, LS, F16, true>(a, split, stream) : few_launch<2, NW, LS, F16, false>(a, split, stream);
    return few_launch<4, NW, LS, F16, false>(a, split, stream);
  };
  switch (waves) {
    case 2: return rows(std::integral_constant<int, 2>{});
    case 3: return rows(std::integral_constant<int, 3>{});
    case 4: return rows(std::integral_constant<int, 4>{});
    case 5: return rows(std::integral_constant<int, 5>{});
    case 6: return rows(std::integral_constant<int, 6>{});
    default: return TBIK_ERR_INVALID;
  }
}

int gemm_tree_few_launch(const WideArgs& a, int leaf_k, bool f16, int waves, int split, hipStream_t stream) {
  if (a.M <= 0 || a.M > 64 || a.N <= 0 || split <= 0 || split > 65535 || (leaf_k != 256 && leaf_k != 128)) return TBIK_ERR_INVALID;
  // the tree of one shard: flb leaves a group, 2^lb groups, and the loads step through exactly K
  if (a.lb < 0 || a.lb > few::LBMAX || a.flb < 1 || a.T != a.flb << a.lb || a.K != a.T * leaf_k) return TBIK_ERR_UNSUPPORTED;
  if (a.ldx >= (1 << 22) || a.ldw >= (1 << 22)) return TBIK_ERR_UNSUPPORTED;  // 32-bit in-tile byte offsets
  if (leaf_k == 256) return f16 ? few_by_shape<4, true>(a, waves, split, stream) : few_by_shape<4, false>(a, waves, split, stream);
  return f16 ? few_by_shape<2, true>(a, waves, split, stream) : few_by_shape<2, false>(a, waves, split, stream);
}

}  // namespace tbik
