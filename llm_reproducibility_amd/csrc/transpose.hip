// Transposing copy of a row-major matrix of 2- or 4-byte elements: out[c][r] = x[r][c], every output row filled up with
// zeros to a given length.  It brings an operand of a matmul that lies the other way round (a row-major right operand, the
// transposed left operand of a weight gradient) into the K-contiguous layout the matmul kernels read; the zeros extend a
// sum over K by exact zero products, so a K of any length reaches the kernels that take whole slices.
//
// Bound: memory, 2 bytes moved per byte.  A wavefront transposes V*8 x V*8 elements (V per 16 bytes: 64x64 or 32x32): a
// lane loads the V rows of one 16-byte column chunk (eight lanes side by side: whole 128-byte lines), transposes its V x V
// block in registers and hands the chunks over through a piece of LDS of its wavefront, swizzled so that neither side
// has bank conflicts, after which eight lanes side by side store whole 128-byte lines.  All V loads are in flight
// together and no wavefront waits for another.
#include "common.h"

namespace tbik {

struct TransposeArgs {
  const uint8_t* x;
  uint8_t* out;
  int64_t ldx, ldo;     // bytes
  int64_t rows, cols;   // of x
  int64_t rows_out;     // elements per output row: rows, then zeros
  int tiles_r;          // tiles along an output row
  int vec;              // x allows 16-byte loads of whole chunks
};

template <int ES>
struct TransposeElem;
template <>
struct TransposeElem<2> { typedef uint16_t type; };
template <>
struct TransposeElem<4> { typedef uint32_t type; };

// V x V block in registers: in[i] = row i (16 bytes), out[i] = column i
__device__ __forceinline__ void transpose_block(const u32x4 (&in)[4], u32x4 (&out)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) out[i][j] = in[j][i];
}
__device__ __forceinline__ void transpose_block(const u32x4 (&in)[8], u32x4 (&out)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)  // elements 2j and 2j + 1 of column i: halves i & 1 of word i / 2 of rows 2j and 2j + 1
      out[i][j] = (i & 1) ? __builtin_amdgcn_perm(in[2 * j + 1][i >> 1], in[2 * j][i >> 1], 0x07060302u)
                          : __builtin_amdgcn_perm(in[2 * j + 1][i >> 1], in[2 * j][i >> 1], 0x05040100u);
}

template <int ES>
__global__ __launch_bounds__(256) void transpose_kernel(const TransposeArgs p) {
  typedef typename TransposeElem<ES>::type elem;
  constexpr int V = 16 / ES, SIDE = 8 * V;
  __shared__ __attribute__((aligned(16))) uint8_t lds[4][SIDE * 128];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // the four wavefronts of a work-group take four tiles side by side along the output rows
  const int64_t tile = (int64_t)blockIdx.x;
  const int64_t r0 = ((tile % p.tiles_r) * 4 + wave) * SIDE;
  const int64_t c0 = (tile / p.tiles_r) * SIDE;
  if (r0 >= p.rows_out) return;
  uint8_t* st = lds[wave];
  {
    const int rg = lane >> 3, cg = lane & 7;   // block of V rows, 16-byte chunk of columns
    const int64_t c = c0 + cg * V;
    u32x4 in[V], tr[V];
    if (p.vec) {   // uniform; cols is then a multiple of V
#pragma unroll
      for (int i = 0; i < V; i++) {
        const int64_t r = r0 + rg * V + i;
        in[i] = u32x4{0u, 0u, 0u, 0u};
        if (r < p.rows && c < p.cols) in[i] = *reinterpret_cast<const u32x4*>(p.x + r * p.ldx + c * ES);
      }
    } else {
#pragma unroll
      for (int i = 0; i < V; i++) {
        const int64_t r = r0 + rg * V + i;
        elem e[V];
#pragma unroll
        for (int j = 0; j < V; j++) {
          e[j] = 0;
          if (r < p.rows && c + j < p.cols) e[j] = *reinterpret_cast<const elem*>(p.x + r * p.ldx + (c + j) * ES);
        }
        __builtin_memcpy(&in[i], e, 16);
      }
    }
    transpose_block(in, tr);
    // column cg * V + i of the tile is LDS row cg * V + i (128 bytes); its chunk rg lies at position rg ^ cg
#pragma unroll
    for (int i = 0; i < V; i++) *reinterpret_cast<u32x4*>(st + (cg * V + i) * 128 + ((rg ^ cg) << 4)) = tr[i];
  }
  // a wavefront reads back only what it wrote itself, and its LDS operations keep their order
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int cl = lane >> 3, pr = lane & 7;
  const int64_t r = r0 + pr * V;
#pragma unroll
  for (int i = 0; i < V; i++) {
    const int col = i * 8 + cl;
    const u32x4 v = *reinterpret_cast<const u32x4*>(st + col * 128 + ((pr ^ (col / V)) << 4));
    if (c0 + col < p.cols && r < p.rows_out) *reinterpret_cast<u32x4*>(p.out + (c0 + col) * p.ldo + r * ES) = v;
  }
}

int transpose_dispatch(const void* x, int64_t ldx, void* out, int64_t ldo, int64_t rows, int64_t cols, int64_t rows_out,
                       int elem_bytes, hipStream_t stream) {
  if (rows < 0 || cols < 0 || rows_out < rows) return TBIK_ERR_INVALID;
  if (elem_bytes != 2 && elem_bytes != 4) return TBIK_ERR_UNSUPPORTED;
  if (cols == 0 || rows_out == 0) return TBIK_OK;
  if ((!x && rows > 0) || !out || (rows > 1 && ldx < cols) || ldo < rows_out) return TBIK_ERR_INVALID;
  const int V = 16 / elem_bytes;
  auto mis = [](const void* q, uintptr_t m) { return (reinterpret_cast<uintptr_t>(q) & m) != 0; };
  if (rows_out % V != 0 || ldo % V != 0 || mis(out, 15) || mis(x, elem_bytes - 1)) return TBIK_ERR_ALIGNMENT;
  const int64_t side = 8 * V, tr = (rows_out + 4 * side - 1) / (4 * side), tc = (cols + side - 1) / side;
  if (tr * tc > 0x7fffffff) return TBIK_ERR_INVALID;
  TransposeArgs a{static_cast<const uint8_t*>(x), static_cast<uint8_t*>(out), ldx * elem_bytes, ldo * elem_bytes, rows, cols, rows_out,
                  (int)tr, !mis(x, 15) && ldx % V == 0 && cols % V == 0};
  const dim3 grid((unsigned)(tr * tc)), block(256);
  if (elem_bytes == 2) hipLaunchKernelGGL(transpose_kernel<2>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(transpose_kernel<4>, grid, block, 0, stream, a);
  return hip_code(hipGetLastError());
}

}  // namespace tbik
