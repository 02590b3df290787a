"""Torch custom ops over the C ABI of libtbik_hip.so.

Each op allocates its output with torch, passes raw device pointers, element strides and the current
HIP stream to one `extern "C"` entry point, and raises on a non-zero return code.  The ops are
registered as `torch.ops.tbik.*` for the GPU device type only; there is no CPU path, CPU tensors raise.

Eager callers reach the same implementation function directly (the dispatcher round trip of a Python
custom op costs ~10 us per call, more than most of these kernels take); under torch.compile the
registered op is used so the call stays a single opaque node.
"""
from __future__ import annotations

import ctypes
import functools
import warnings
from typing import List, Optional

import torch

from . import _lib

_DTYPE_CODE = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    """The current stream of the tensor's device as a raw handle.  The private accessor (the one torch's own compiled code
    uses) returns the handle without building a Stream object: 0.3 us instead of 3 us of host time per launch."""
    if _raw_stream is not None and t.device.index is not None:
        return _raw_stream(t.device.index)
    return torch.cuda.current_stream(t.device).cuda_stream


_fast_module = None


class _NoFast:
    """Stands in for the extension where there is none to use: every call goes the way written out here."""
    rms_norm = add_rms_norm = silu_mul = mean_last = log_softmax = staticmethod(lambda *args: None)


def _fast():
    """The extension with the common calls of the row-wise operators (csrc_host/fast_ops.cpp): each gives the result, or None
    for a call that is not the plain case, which then goes the way written out here.  The same kernels run either way, so
    one that is missing, or built for another library or torch, costs host time only: a warning, once."""
    global _fast_module
    if _fast_module is None:
        _lib.lib()   # a missing library is reported as such
        why = None
        try:
            from . import _fast as module
        except ImportError as e:
            why = f"does not load ({e})"
        else:
            built_for = getattr(module, "built_for", "nothing it tells")
            if built_for != _lib.fast_built_for():
                why = f"was built for {built_for}, this is {_lib.fast_built_for()}"
        if why:
            warnings.warn(f"the host extension llm_reproducibility_amd._fast {why}: row-wise operators take a slower way to the same "
                          "kernels; run `python -m llm_reproducibility_amd.build`", RuntimeWarning, stacklevel=2)
            module = _NoFast
        _fast_module = module
    return _fast_module


def _require_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("tbik ops run on the GPU only (HIP kernels); got a tensor on " + str(t.device))


def _aligned16(t: torch.Tensor) -> bool:
    return t.data_ptr() % 16 == 0


def _is_f16(*tensors) -> bool:
    """True for float16 operands, False for bfloat16; every operand must have the same one of the two."""
    dt = tensors[0].dtype
    same = dt is torch.bfloat16 or dt is torch.float16
    for t in tensors:
        if t is not None and t.dtype is not dt:
            same = False
    if not same:
        dts = {t.dtype for t in tensors if t is not None}
        raise NotImplementedError(f"16-bit GEMM kernels take all-bfloat16 or all-float16 operands, got {sorted(map(str, dts))}")
    return dt is torch.float16


def _k_across(t: torch.Tensor) -> bool:
    """True for a matrix whose columns are contiguous and whose rows are not, the transposed view of a row-major one, in an
    element size that the transposing copy takes (other types are refused further on, as what they are)."""
    (rows, cols), (s0, s1) = t.shape, t.stride()
    return s0 == 1 and s1 != 1 and rows > 1 and cols > 1 and s1 >= rows and t.element_size() in (2, 4)


def _transposed(t: torch.Tensor, k: int):
    """(copy of the `_k_across` matrix t with contiguous rows, its leading dimension): one pass of the transposing copy
    kernel, the rows extended by zeros to k elements (a multiple of 16 bytes).  4.2 - 5.0 TB/s, where the library's
    strided copy moves 1 TB/s in 16 bits and 2 in 32 ([12288,4096] bf16: 45 us against 196)."""
    R, C = t.shape
    out = torch.empty((R, k), device=t.device, dtype=t.dtype)
    rc = _lib.lib().bi_transpose(t.data_ptr(), t.stride(1), out.data_ptr(), k, C, R, k, t.element_size(), _stream(t))
    _lib.check(rc, "bi_transpose")
    return out, k


def _k_rows(t: torch.Tensor, k: int):
    """(tensor, leading dimension) of t with contiguous rows, extended by zero columns to k."""
    if _k_across(t):
        return _transposed(t, k)
    p = torch.nn.functional.pad(t, (0, k - t.shape[1]))
    return p, p.stride(0)


def _rows_f32(t: torch.Tensor):
    """fp32 operand with a contiguous last dim, 16-byte aligned rows (leading dimension a multiple of 4)."""
    ok = t.stride(1) == 1 and _aligned16(t) and (t.shape[0] == 1 or (t.stride(0) >= t.shape[1] and t.stride(0) % 4 == 0))
    if ok:
        return t, (t.shape[1] if t.shape[0] == 1 else t.stride(0))
    if _k_across(t):
        return _transposed(t, (t.shape[1] + 3) // 4 * 4)
    c = t.contiguous()
    if not _aligned16(c) or c.shape[1] % 4 != 0:
        c = torch.nn.functional.pad(c, (0, (-c.shape[1]) % 4))[:, : t.shape[1]] if c.shape[1] % 4 else c.clone()
    return c, c.stride(0)


def _gemm_f32(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], leaf_k: int, tree: bool) -> torch.Tensor:
    M, K = A.shape
    N = B.shape[1]
    if K % 16 != 0:  # only the single-accumulator form gets here: zero columns do not change a sequential sum
        K += (-K) % 16
        a, lda = _k_rows(A, K)
        w, ldw = _k_rows(B.t(), K)
    else:
        a, lda = _rows_f32(A)
        w, ldw = _rows_f32(B.t())
    b = None if bias is None else bias.contiguous()
    C = torch.empty((M, N), device=A.device, dtype=torch.float32)
    L = _lib.lib()
    if tree:
        rc = L.tbik_gemm_f32(a.data_ptr(), lda, w.data_ptr(), 1, ldw, C.data_ptr(), C.stride(0), M, N, K, leaf_k,
                             None if b is None else b.data_ptr(), _stream(A))
    else:
        rc = L.bi_gemm_f32(a.data_ptr(), lda, w.data_ptr(), 1, ldw, C.data_ptr(), C.stride(0), M, N, K,
                           None if b is None else b.data_ptr(), _stream(A))
    _lib.check(rc, "tbik_gemm_f32" if tree else "bi_gemm_f32")
    return C


def _rows16(t: torch.Tensor):
    """(tensor, leading dimension) with a contiguous last dim and 16-byte aligned rows; copies if needed."""
    (rows, cols), (s0, s1) = t.shape, t.stride()
    if s1 == 1 and cols % 8 == 0 and _aligned16(t):
        if rows == 1:
            return t, cols
        if s0 >= cols and s0 % 8 == 0:
            return t, s0
    if _k_across(t):
        return _transposed(t, (t.shape[1] + 7) // 8 * 8)
    c = t.contiguous()
    if not _aligned16(c):
        c = c.clone()
    return c, c.shape[1]


def _flat_rows16(t: torch.Tensor):
    """`_rows16` of t as a matrix of its last dimension.  A matrix is taken as it is: a reshape to its own shape costs
    0.8 us of host time, and the call of a norm of a few rows is nothing but host time (four of them fewer, the leading
    dimensions read once: 15.6 us -> 10.4 us)."""
    return _rows16(t if t.dim() == 2 else t.reshape(-1, t.shape[-1]))


def _unflat(out: torch.Tensor, shape) -> torch.Tensor:
    return out if len(shape) == 2 else out.reshape(shape)


# Where a row-major [K,N] operand that the K-major kernels do not take (`_bi_gemm_kmajor`: odd columns, a K that is no multiple of
# 64, or no gain; `_tree_operand`: columns that are no multiple of eight, 256 leaves and more) is repacked into the native [N,K]
# layout instead of being consumed in place.  In place it runs on the 64-row tiled kernels; a repack is one pass of the transposing copy kernel (23 us for 4096 x 4096 in 16 bits,
# 45 us for 12288 x 4096) and then whatever kernel is best.  Same bits either way.  Measured on MI355X, us in place against repacked:
#   tree matmul: in place cuts K and holds out until its 64-row tiles fill a second round of the chip, that is up to 128
#     rows (12288 x 4096: 68 against 73; at 192 rows 99 against 79, at 1024 448 against 164), later for small matrices
#     (2048 x 1536: 256 rows 16 against 20, 384 rows 27 against 21; 1024 x 1024: 1024 rows 16.3 against 17.4, 1536 rows 26.5
#     against 18.1; 512 x 1536: 1536 rows, 288 tiles, 22.8 against 14.4): bounds on rows * K * N and on the tiles.
#   single-accumulator mm: in place cannot cut K, so a call takes as long as one chain per round of 512 work-groups (two on
#     a CU), whatever it fills them with; narrow matrices are repacked (4096 x 4096: 88 against 27 at one row, 77 against 34 at
#     64), wide ones not while they are one round (12288 x 16384: 220 against 273 at 64 rows, 248 against 318 at 256; 4096 x
#     24576: 93 against 123 at 128 rows, 158 against 138 at 160).  K, the rounds and, for a K that is no multiple of 64, the type (fp16
#     has the large tiles of bf16 for whole slices only) move the line, so both times are estimated.
#   Both estimates are of whole column tiles (N a multiple of 128, of 64 up to 16 rows): for the mm, 1 .. 3072 rows, K = 512 .. 25600, N =
#     512 .. 48000 in both types, the choice is 0.5 % from the better of the two on average there and 12 % at worst (62 points).  A
#     last tile that is not whole, which every tree operand has that comes here, costs the 64-row tiles two to four times the time, which the
#     estimates do not know: where such an operand stays in place a repack would nearly always be ahead, 1.8 times on average.
_TREE_IN_PLACE_MACS = 416 * 2048 * 1536


def _consumed_in_place(rows: int, K: int, N: int, tree: bool, f16: bool = False) -> bool:
    tiles = -(-rows // 64) * -(-N // 128)
    if tree:
        return rows <= 128 or (rows * K * N < _TREE_IN_PLACE_MACS and tiles <= 256)
    groups = -(-N // 64) if rows <= 16 else tiles
    in_place = (7.0 + 0.0222 * K) * max(1, -(-groups // 512))
    copied = 4.0 * K * N    # bytes; up to 256 MB the cache behind the L2s holds them
    product = max(K * N / 3.5e6, 0.0048 * K if rows > 64 else 0.0)
    if f16 and rows > 64 and K % 64:
        product = max(product, 0.0098 * K * -(-(-(-rows // 128) * -(-N // 128)) // 256))
    else:
        product = max(product, rows * K * N / 0.72e9)
    return in_place < 11.8 + copied / (4.1e6 if copied <= 256e6 else 3.3e6) + product


def _weight_operand(B: torch.Tensor, rows: int = 0, tree: bool = True):
    """How a [K,N] operand is handed to the kernels: (tensor whose data_ptr is passed, ldb_k, ldb_n).

    `weight.t()` of an nn.Linear weight ([N,K], K contiguous) is the native layout (ldb_k = 1), used without a copy; a
    row-major [K,N] operand (N contiguous: a plain `x @ B`) is consumed in place too (ldb_n = 1) unless a repack into
    the native layout pays for this many `rows`.  Anything else -- neither dimension contiguous, rows not 16-byte
    aligned -- is repacked as well."""
    (K, N), (s0, s1) = B.shape, B.stride()
    if s0 == 1 and _aligned16(B) and K % 8 == 0 and (N == 1 or (s1 >= K and s1 % 8 == 0)):
        return B, 1, (K if N == 1 else s1)
    if s1 == 1 and _aligned16(B) and s0 >= N and s0 % 8 == 0 and _consumed_in_place(rows, K, N, tree, B.dtype is torch.float16):
        return B, s0, 1
    w, ldw = _rows16(B.t())
    return w, 1, ldw


def _tree_operand(B: torch.Tensor, rows: int, leaf_k: int):
    """`_weight_operand` of a tree matmul: a row-major operand that the library can read K-major (whole chunks of eight columns,
    and a tree that those tiles hold: fewer than 256 leaves always are) stays in place where it says that this pays, and is
    repacked where it does not."""
    (K, N), (s0, s1) = B.shape, B.stride()
    if s1 == 1 and N % 8 == 0 and _aligned16(B) and s0 >= N and s0 % 8 == 0 and K < 256 * leaf_k:
        if _lib.lib().tbik_gemm_rowmajor_b_pays(rows, N, K, leaf_k):
            return B, s0, 1
        w, ldw = _rows16(B.t())
        return w, 1, ldw
    return _weight_operand(B, rows, True)


# --------------------------------------------------------------------------------------------
# tree-ordered GEMM
# --------------------------------------------------------------------------------------------
def _gemm_tree_impl(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], leaf_k: int) -> torch.Tensor:
    _require_gpu(A, B, bias)
    if A.dtype == torch.float32 and B.dtype == torch.float32 and (bias is None or bias.dtype == torch.float32):
        return _gemm_f32(A, B, bias, leaf_k, True)
    M, K = A.shape
    N = B.shape[1]
    a, lda = _rows16(A)
    w, ldb_k, ldb_n = _tree_operand(B, M, leaf_k)
    b = None if bias is None else bias.contiguous()
    f16 = _is_f16(A, B, bias)
    C = torch.empty((M, N), device=A.device, dtype=A.dtype)
    L = _lib.lib()
    if ldb_k != 1:
        ws_bytes = L.tbik_gemm_workspace_bytes_rowmajor_b(M, N, K, leaf_k, int(f16))
    else:
        ws_bytes = (L.tbik_gemm_f16_workspace_bytes if f16 else L.tbik_gemm_workspace_bytes)(M, N, K, leaf_k)
    ws = torch.empty(ws_bytes, device=A.device, dtype=torch.uint8) if ws_bytes else None
    rc = (L.tbik_gemm_f16 if f16 else L.tbik_gemm_bf16)(a.data_ptr(), lda, w.data_ptr(), ldb_k, ldb_n, C.data_ptr(), C.stride(0),
                          M, N, K, leaf_k, None if b is None else b.data_ptr(),
                          None if ws is None else ws.data_ptr(), ws_bytes, _stream(A))
    _lib.check(rc, "tbik_gemm_bf16")
    return C


_gemm_tree_op = torch.library.custom_op("tbik::gemm_tree", _gemm_tree_impl, mutates_args=(), device_types="cuda")


def gemm_tree(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], leaf_k: int) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _gemm_tree_op(A, B, bias, leaf_k)
    return _gemm_tree_impl(A, B, bias, leaf_k)


@_gemm_tree_op.register_fake
def _(A, B, bias, leaf_k):
    return A.new_empty((A.shape[0], B.shape[1]))


def _check_sharded(A: torch.Tensor, W: torch.Tensor) -> None:
    """K is taken from A alone: a W of other columns would be read in part, or behind its rows."""
    if A.dim() != 2 or W.dim() != 2 or A.shape[1] != W.shape[1]:
        raise ValueError(f"gemm_tree_sharded takes A [M,K] and W [N,K], got {tuple(A.shape)} and {tuple(W.shape)}")
    if A.device != W.device:
        raise ValueError(f"gemm_tree_sharded takes operands on one device, got {A.device} and {W.device}")


def _gemm_tree_sharded_impl(A: torch.Tensor, W: torch.Tensor, leaf_k: int, shards: int) -> torch.Tensor:
    _check_sharded(A, W)
    _require_gpu(A, W)
    M, K = A.shape
    N = W.shape[0]
    f16 = _is_f16(A, W)
    L = _lib.lib()
    if not L.tbik_gemm_sharded_pays(M, N, K, leaf_k, shards, int(f16)):
        ks = K // shards
        return _tree_combine_impl([_gemm_tree_impl(A[:, r * ks:(r + 1) * ks], W[:, r * ks:(r + 1) * ks].t(), None, leaf_k) for r in range(shards)])
    a, lda = _rows16(A)
    w, ldw = _rows16(W)
    C = torch.empty((M, N), device=A.device, dtype=A.dtype)
    ws_bytes = L.tbik_gemm_sharded_workspace_bytes(M, N, K, leaf_k, shards, int(f16))
    ws = torch.empty(ws_bytes, device=A.device, dtype=torch.uint8) if ws_bytes else None
    rc = L.tbik_gemm_sharded(a.data_ptr(), lda, w.data_ptr(), ldw, C.data_ptr(), C.stride(0), M, N, K, leaf_k, shards, int(f16), None,
                             None if ws is None else ws.data_ptr(), ws_bytes, _stream(A))
    _lib.check(rc, "tbik_gemm_sharded")
    return C


_gemm_tree_sharded_op = torch.library.custom_op("tbik::gemm_tree_sharded", _gemm_tree_sharded_impl, mutates_args=(), device_types="cuda")


def gemm_tree_sharded(A: torch.Tensor, W: torch.Tensor, leaf_k: int, shards: int) -> torch.Tensor:
    """The products of all `shards` ranks of a row-split layer (weight W [N,K], 16 bits) and the shard tree over them: one grid
    and one combine, or, where the library expects more of it, a `gemm_tree` per rank and `tree_combine`; the same bits.  shards: a power of two up to 32."""
    if torch.compiler.is_compiling():
        return _gemm_tree_sharded_op(A, W, leaf_k, shards)
    return _gemm_tree_sharded_impl(A, W, leaf_k, shards)


@_gemm_tree_sharded_op.register_fake
def _(A, W, leaf_k, shards):
    _check_sharded(A, W)
    return A.new_empty((A.shape[0], W.shape[0]))


def _tree_combine_impl(parts: List[torch.Tensor]) -> torch.Tensor:
    _require_gpu(*parts)
    ps = [p.contiguous() for p in parts]
    out = torch.empty_like(ps[0])
    arr = (ctypes.c_void_p * len(ps))(*[p.data_ptr() for p in ps])
    L = _lib.lib()
    if ps[0].dtype == torch.float32:
        if any(p.dtype != torch.float32 for p in ps):
            raise NotImplementedError("tree_combine takes partials of one dtype")
        fn = L.tbik_tree_combine_f32
    else:
        fn = L.tbik_tree_combine_f16 if _is_f16(*ps) else L.tbik_tree_combine_bf16
    rc = fn(arr, len(ps), out.data_ptr(), out.numel(), _stream(out))
    _lib.check(rc, "tbik_tree_combine")
    return out


_tree_combine_op = torch.library.custom_op("tbik::tree_combine", _tree_combine_impl, mutates_args=(), device_types="cuda")


def tree_combine(parts: List[torch.Tensor]) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _tree_combine_op(parts)
    return _tree_combine_impl(parts)


@_tree_combine_op.register_fake
def _(parts):
    return torch.empty_like(parts[0])


# --------------------------------------------------------------------------------------------
# batch-invariant ops
# --------------------------------------------------------------------------------------------
def _bi_gemm_kmajor(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], f16: bool) -> Optional[torch.Tensor]:
    """A @ B in 16 bits with a row-major B (and, in a weight gradient, an A whose columns are contiguous) read in place; None
    where the library prefers copies or an operand lies otherwise.  Same bits either way."""
    (M, K), N = A.shape, B.shape[1]
    across = _k_across(A)
    lda, ldb = A.stride(1 if across else 0), B.stride(0)
    if M == 1 and not across:
        lda = K
    if not ((across and M % 8 == 0) or (A.stride(1) == 1 and K % 64 == 0 and lda >= K)):
        return None
    if K == 1 or ldb < N or ldb % 8 or lda % 8 or not _aligned16(A) or not _aligned16(B):
        return None
    b = None if bias is None else bias.contiguous()
    C = torch.empty((M, N), device=A.device, dtype=A.dtype)
    L = _lib.lib()
    rc = (L.bi_gemm_kmajor_f16 if f16 else L.bi_gemm_kmajor_bf16)(
        A.data_ptr(), lda, int(across), B.data_ptr(), ldb, C.data_ptr(), C.stride(0), M, N, K,
        None if b is None else b.data_ptr(), _stream(A))
    if rc == _lib.TBIK_ERR_UNSUPPORTED:
        return None
    _lib.check(rc, "bi_gemm_kmajor")
    return C


def _bi_gemm_impl(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    _require_gpu(A, B, bias)
    if A.dtype == torch.float32 and B.dtype == torch.float32 and (bias is None or bias.dtype == torch.float32):
        return _gemm_f32(A, B, bias, 0, False)
    M, K = A.shape
    N = B.shape[1]
    f16 = _is_f16(A, B, bias)
    if B.stride(1) == 1 and N % 8 == 0:
        C = _bi_gemm_kmajor(A, B, bias, f16)
        if C is not None:
            return C
    if K % 8 != 0 or (K % 64 != 0 and _k_across(A) and _k_across(B.t())):
        # zero columns do not change a sequential fp32 accumulation.  A K that no kernel takes is extended, and so is one
        # that only the small-tile kernel takes when both operands are copied anyway (a weight gradient, whose K is
        # the number of tokens): to whole slices of 64, which every kernel takes
        K += (-K) % 64
        a, lda = _k_rows(A, K)
        w, ldb_n = _k_rows(B.t(), K)
        ldb_k = 1
    else:
        a, lda = _rows16(A)
        w, ldb_k, ldb_n = _weight_operand(B, M, False)
    b = None if bias is None else bias.contiguous()
    C = torch.empty((M, N), device=A.device, dtype=A.dtype)
    L = _lib.lib()
    rc = (L.bi_gemm_f16 if f16 else L.bi_gemm_bf16)(a.data_ptr(), lda, w.data_ptr(), ldb_k, ldb_n, C.data_ptr(), C.stride(0),
                                 M, N, K, None if b is None else b.data_ptr(), _stream(A))
    _lib.check(rc, "bi_gemm")
    return C


_bi_gemm_op = torch.library.custom_op("tbik::bi_gemm", _bi_gemm_impl, mutates_args=(), device_types="cuda")


def bi_gemm(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _bi_gemm_op(A, B, bias)
    return _bi_gemm_impl(A, B, bias)


@_bi_gemm_op.register_fake
def _(A, B, bias):
    return A.new_empty((A.shape[0], B.shape[1]))


def _bi_rmsnorm_impl(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    _require_gpu(x, weight)
    hidden = x.shape[-1]
    x2, ldx = _flat_rows16(x)
    rows = x2.shape[0]
    out = torch.empty((rows, hidden), device=x.device, dtype=x.dtype)
    w = None if weight is None else weight.contiguous()
    L = _lib.lib()
    rc = (L.bi_rmsnorm_f16 if _is_f16(x, weight) else L.bi_rmsnorm_bf16)(x2.data_ptr(), ldx, None, 0, None if w is None else w.data_ptr(),
                                    out.data_ptr(), hidden, None, 0, rows, hidden, eps, _stream(x))
    _lib.check(rc, "bi_rmsnorm")
    return _unflat(out, x.shape)


_bi_rmsnorm_op = torch.library.custom_op("tbik::bi_rmsnorm", _bi_rmsnorm_impl, mutates_args=(), device_types="cuda")


def bi_rmsnorm(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _bi_rmsnorm_op(x, weight, eps)
    out = (_fast_module or _fast()).rms_norm(x, weight, eps)
    return _bi_rmsnorm_impl(x, weight, eps) if out is None else out


@_bi_rmsnorm_op.register_fake
def _(x, weight, eps):
    return torch.empty_like(x)


def _bi_add_rmsnorm_impl(x: torch.Tensor, residual: torch.Tensor, weight: Optional[torch.Tensor],
                        eps: float) -> List[torch.Tensor]:
    _require_gpu(x, residual, weight)
    hidden = x.shape[-1]
    x2, ldx = _flat_rows16(x)
    r2, ldr = _rows16(residual if residual.dim() == 2 and residual.shape[1] == hidden else residual.reshape(-1, hidden))
    rows = x2.shape[0]
    out = torch.empty((rows, hidden), device=x.device, dtype=x.dtype)
    rout = torch.empty_like(out)
    w = None if weight is None else weight.contiguous()
    L = _lib.lib()
    rc = (L.bi_rmsnorm_f16 if _is_f16(x, residual, weight) else L.bi_rmsnorm_bf16)(x2.data_ptr(), ldx, r2.data_ptr(), ldr,
                                    None if w is None else w.data_ptr(), out.data_ptr(), hidden,
                                    rout.data_ptr(), hidden, rows, hidden, eps, _stream(x))
    _lib.check(rc, "bi_rmsnorm")
    return [_unflat(out, x.shape), _unflat(rout, x.shape)]


_bi_add_rmsnorm_op = torch.library.custom_op("tbik::bi_add_rmsnorm", _bi_add_rmsnorm_impl, mutates_args=(), device_types="cuda")


def bi_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor, weight: Optional[torch.Tensor],
                        eps: float) -> List[torch.Tensor]:
    if torch.compiler.is_compiling():
        return _bi_add_rmsnorm_op(x, residual, weight, eps)
    out = (_fast_module or _fast()).add_rms_norm(x, residual, weight, eps)
    return _bi_add_rmsnorm_impl(x, residual, weight, eps) if out is None else out


@_bi_add_rmsnorm_op.register_fake
def _(x, residual, weight, eps):
    return [torch.empty_like(x), torch.empty_like(x)]


def _bi_log_softmax_impl(x: torch.Tensor, write_softmax: bool, to_float: bool) -> torch.Tensor:
    """log_softmax (or softmax) over the last dimension of an fp32 / bf16 / fp16 tensor, in the input's dtype or,
    with `to_float`, in fp32; the kernel reads the input dtype itself."""
    _require_gpu(x)
    if x.dtype not in _DTYPE_CODE:
        raise NotImplementedError(f"bi_log_softmax: unsupported dtype {x.dtype}")
    cols = x.shape[-1]
    x2 = x.reshape(-1, cols)
    if x2.stride(1) != 1 or (x2.shape[0] > 1 and x2.stride(0) < cols):
        x2 = x2.contiguous()
    rows = x2.shape[0]
    out_dtype = torch.float32 if to_float else x.dtype
    out = torch.empty((rows, cols), device=x.device, dtype=out_dtype)
    L = _lib.lib()
    nws = L.bi_log_softmax_workspace_bytes(rows, cols)
    ws = torch.empty((nws + 3) // 4, device=x.device, dtype=torch.float32) if nws else None
    rc = L.bi_log_softmax(x2.data_ptr(), x2.stride(0) if rows > 1 else cols, _DTYPE_CODE[x.dtype], out.data_ptr(),
                          out.stride(0), _DTYPE_CODE[out_dtype], rows, cols, None if ws is None else ws.data_ptr(), nws,
                          int(write_softmax), _stream(x))
    _lib.check(rc, "bi_log_softmax")
    return out.reshape(x.shape)


_bi_log_softmax_op = torch.library.custom_op("tbik::bi_log_softmax", _bi_log_softmax_impl, mutates_args=(), device_types="cuda")


def bi_log_softmax(x: torch.Tensor, write_softmax: bool, to_float: bool = False) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _bi_log_softmax_op(x, write_softmax, to_float)
    out = (_fast_module or _fast()).log_softmax(x, write_softmax, to_float)
    return _bi_log_softmax_impl(x, write_softmax, to_float) if out is None else out


@_bi_log_softmax_op.register_fake
def _(x, write_softmax, to_float):
    return torch.empty_like(x, dtype=torch.float32 if to_float else x.dtype)


def bi_log_softmax_f32(x: torch.Tensor, write_softmax: bool) -> torch.Tensor:
    """fp32 in, fp32 out (kept for callers of the earlier name)."""
    return bi_log_softmax(x.float(), write_softmax)


def _bi_mean_dim_impl(x: torch.Tensor, dim: int, keepdim: bool) -> torch.Tensor:
    _require_gpu(x)
    if x.dtype not in _DTYPE_CODE:
        raise NotImplementedError(f"bi_mean_dim: unsupported dtype {x.dtype}")
    dim = dim % x.ndim
    shape = list(x.shape)
    outer = 1
    for s in shape[:dim]:
        outer *= s
    n = shape[dim]
    inner = 1
    for s in shape[dim + 1:]:
        inner *= s
    xc = x.contiguous()
    out_shape = shape[:dim] + ([1] if keepdim else []) + shape[dim + 1:]
    out = torch.empty(out_shape, device=x.device, dtype=x.dtype)
    rc = _lib.lib().bi_mean_dim(xc.data_ptr(), out.data_ptr(), outer, n, inner, _DTYPE_CODE[x.dtype], _stream(x))
    _lib.check(rc, "bi_mean_dim")
    return out


_bi_mean_dim_op = torch.library.custom_op("tbik::bi_mean_dim", _bi_mean_dim_impl, mutates_args=(), device_types="cuda")


def bi_mean_dim(x: torch.Tensor, dim: int, keepdim: bool) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _bi_mean_dim_op(x, dim, keepdim)
    out = (_fast_module or _fast()).mean_last(x, keepdim) if dim == -1 or dim == x.ndim - 1 else None
    return _bi_mean_dim_impl(x, dim, keepdim) if out is None else out


@_bi_mean_dim_op.register_fake
def _(x, dim, keepdim):
    dim = dim % x.ndim
    shape = list(x.shape)
    out_shape = shape[:dim] + ([1] if keepdim else []) + shape[dim + 1:]
    return x.new_empty(out_shape)


# --------------------------------------------------------------------------------------------
# fixed-order attention
# --------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=1024)
def _attention_workspace_bytes(*shape: int) -> int:
    """A function of five numbers, asked of the library once: 0.3 of the 9.4 us that a short decode call takes the host."""
    return _lib.lib().bi_attention_workspace_bytes(*shape)


def _attention_workspace(batch: int, max_q_len: int, q_heads: int, kv_heads: int, max_len: int, device):
    """(scratch for the chunks of long caches that several work-groups share, its bytes); (None, 0) where none is used."""
    n = _attention_workspace_bytes(batch, max_q_len, q_heads, kv_heads, max_len)
    return (torch.empty(n, device=device, dtype=torch.uint8), n) if n else (None, 0)


def _bi_attention_bf16_impl(q: torch.Tensor, k_cache: torch.Tensor, vt_cache: torch.Tensor, q_start: torch.Tensor,
                            q_len: torch.Tensor, ctx_len: torch.Tensor, max_q_len: int, scale: float) -> torch.Tensor:
    _require_gpu(q, k_cache, vt_cache, q_start, q_len, ctx_len)
    tokens, q_heads, head_dim = q.shape
    batch, kv_heads, max_len, _ = k_cache.shape
    assert vt_cache.shape == (batch, kv_heads, head_dim, max_len)
    assert q.dtype == torch.bfloat16 and k_cache.dtype == torch.bfloat16 and vt_cache.dtype == torch.bfloat16
    assert q_start.dtype == torch.int32 and q_len.dtype == torch.int32 and ctx_len.dtype == torch.int32
    q = q.contiguous()
    assert k_cache.is_contiguous() and vt_cache.is_contiguous()
    out = torch.empty_like(q)
    ws, ws_bytes = _attention_workspace(batch, max_q_len, q_heads, kv_heads, max_len, q.device)
    rc = _lib.lib().bi_attention_ws_bf16(q.data_ptr(), k_cache.data_ptr(), vt_cache.data_ptr(), out.data_ptr(),
                                         q_start.data_ptr(), q_len.data_ptr(), ctx_len.data_ptr(), batch, max_q_len,
                                         q_heads, kv_heads, head_dim, max_len, scale,
                                         None if ws is None else ws.data_ptr(), ws_bytes, _stream(q))
    _lib.check(rc, "bi_attention_ws_bf16")
    return out


_bi_attention_bf16_op = torch.library.custom_op("tbik::bi_attention_bf16", _bi_attention_bf16_impl, mutates_args=(),
                                                device_types="cuda")


def bi_attention_bf16(q: torch.Tensor, k_cache: torch.Tensor, vt_cache: torch.Tensor, q_start: torch.Tensor,
                      q_len: torch.Tensor, ctx_len: torch.Tensor, max_q_len: int, scale: float) -> torch.Tensor:
    if torch.compiler.is_compiling():
        return _bi_attention_bf16_op(q, k_cache, vt_cache, q_start, q_len, ctx_len, max_q_len, scale)
    return _bi_attention_bf16_impl(q, k_cache, vt_cache, q_start, q_len, ctx_len, max_q_len, scale)


@_bi_attention_bf16_op.register_fake
def _(q, k_cache, vt_cache, q_start, q_len, ctx_len, max_q_len, scale):
    return torch.empty_like(q)


# --------------------------------------------------------------------------------------------
# gated activation in front of down_proj
# --------------------------------------------------------------------------------------------
def _bi_silu_mul_impl(gate_up: torch.Tensor) -> torch.Tensor:
    _require_gpu(gate_up)
    f16 = _is_f16(gate_up)
    two_i = gate_up.shape[-1]
    if two_i % 16 != 0:
        raise ValueError(f"bi_silu_mul: last dimension {two_i} must be a multiple of 16")
    inter = two_i // 2
    g2, ld = _flat_rows16(gate_up)
    rows = g2.shape[0]
    out = torch.empty((rows, inter), device=gate_up.device, dtype=gate_up.dtype)
    L = _lib.lib()
    rc = (L.bi_silu_mul_f16 if f16 else L.bi_silu_mul_bf16)(g2.data_ptr(), ld, out.data_ptr(), inter, rows, inter, _stream(gate_up))
    _lib.check(rc, "bi_silu_mul")
    return _unflat(out, (*gate_up.shape[:-1], inter))


_bi_silu_mul_op = torch.library.custom_op("tbik::bi_silu_mul", _bi_silu_mul_impl, mutates_args=(), device_types="cuda")


def bi_silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """act = silu(gate_up[..., :I]) * gate_up[..., I:] (I = half the last dimension), fused, bf16."""
    if torch.compiler.is_compiling():
        return _bi_silu_mul_op(gate_up)
    out = (_fast_module or _fast()).silu_mul(gate_up)
    return _bi_silu_mul_impl(gate_up) if out is None else out


@_bi_silu_mul_op.register_fake
def _(gate_up):
    return gate_up.new_empty((*gate_up.shape[:-1], gate_up.shape[-1] // 2))


# --------------------------------------------------------------------------------------------
# one-launch compositions for decode-sized batches (bit-identical to the two-launch forms they fall back to)
# --------------------------------------------------------------------------------------------
# Shapes for which a one-launch entry point answered 'unsupported': whether it applies depends on the shape alone (what
# depends on strides is asked before the call), so the next call of the same shape goes to the separate calls at once (no
# output allocated for a call that will not run).  Row counts of a serving program are many: the set starts anew when full.
_declined: set = set()
_DECLINED_MAX = 4096
_FAR_ROWS = 1 << 22   # row stride from which the 256-row tiles' 32-bit byte offsets do not reach


def _decline(key) -> None:
    if len(_declined) >= _DECLINED_MAX:
        _declined.clear()
    _declined.add(key)


def rmsnorm_gemm(x: torch.Tensor, norm_weight: Optional[torch.Tensor], eps: float, residual: Optional[torch.Tensor],
                 B: torch.Tensor, bias: Optional[torch.Tensor] = None):
    """(bi_gemm(rms_norm(x [+ residual]) * norm_weight, B) (+ bias), new residual or None).

    One launch (`bi_rmsnorm_gemm_bf16`: the matmul normalises the activations while it stages them) for a few bf16 rows
    against an nn.Linear weight handed over as `weight.t()`; the two launches otherwise.  Same bits either way."""
    _require_gpu(x, norm_weight, residual, B, bias)
    M, K = x.shape
    N = B.shape[1]
    fusable = (x.dtype == torch.bfloat16 and B.dtype == torch.bfloat16 and M * K <= 32768 and K <= 8192 and K % 32 == 0
               and B.stride(0) == 1 and not torch.compiler.is_compiling() and ("norm_mm", M, N, K) not in _declined)
    if fusable:
        x2, ldx = _rows16(x)
        r2, ldr = (None, 0) if residual is None else _rows16(residual)
        w, ldb_k, ldb_n = _weight_operand(B)
        nw = None if norm_weight is None else norm_weight.contiguous()
        b = None if bias is None else bias.contiguous()
        C = torch.empty((M, N), device=x.device, dtype=x.dtype)
        rout = None if residual is None else torch.empty((M, K), device=x.device, dtype=x.dtype)
        rc = _lib.lib().bi_rmsnorm_gemm_bf16(x2.data_ptr(), ldx, None if r2 is None else r2.data_ptr(), ldr,
                                             None if nw is None else nw.data_ptr(), eps,
                                             None if rout is None else rout.data_ptr(), K, w.data_ptr(), ldb_k, ldb_n,
                                             C.data_ptr(), C.stride(0), M, N, K, None if b is None else b.data_ptr(), _stream(x))
        if rc == _lib.TBIK_OK:
            return C, rout
        if rc != _lib.TBIK_ERR_UNSUPPORTED:
            _lib.check(rc, "bi_rmsnorm_gemm_bf16")
        _decline(("norm_mm", M, N, K))
    if residual is None:
        h, rout = bi_rmsnorm(x, norm_weight, eps), None
    else:
        h, rout = bi_add_rmsnorm(x, residual, norm_weight, eps)
    return bi_gemm(h, B, bias), rout


def gemm_tree_silu_mul(gate: torch.Tensor, up: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], leaf_k: int) -> torch.Tensor:
    """gemm_tree(silu(gate) * up, B, bias, leaf_k) for the two halves (or a K shard of both halves) of a merged gate/up
    projection: column slices of one tensor, same row stride.

    One launch (`tbik_gemm_silu_mul_bf16`) for a few bf16 rows, the activation kernel followed by the tree matmul
    otherwise.  Same bits either way."""
    _require_gpu(gate, up, B, bias)
    M, K = gate.shape
    N = B.shape[1]
    fusable = (gate.dtype == torch.bfloat16 and B.dtype == torch.bfloat16 and M <= 4 and up.shape == gate.shape
               and gate.stride(1) == 1 and up.stride(1) == 1 and gate.stride(0) == up.stride(0) and gate.stride(0) % 8 == 0
               and _aligned16(gate) and _aligned16(up) and B.stride(0) == 1 and not torch.compiler.is_compiling()
               and ("silu_tree", M, N, K, leaf_k) not in _declined)
    if fusable:
        w, ldb_k, ldb_n = _weight_operand(B)
        b = None if bias is None else bias.contiguous()
        C = torch.empty((M, N), device=gate.device, dtype=gate.dtype)
        rc = _lib.lib().tbik_gemm_silu_mul_bf16(gate.data_ptr(), up.data_ptr(), gate.stride(0) if M > 1 else max(gate.stride(0), K),
                                                w.data_ptr(), ldb_k, ldb_n, C.data_ptr(), C.stride(0), M, N, K, leaf_k,
                                                None if b is None else b.data_ptr(), _stream(gate))
        if rc == _lib.TBIK_OK:
            return C
        if rc != _lib.TBIK_ERR_UNSUPPORTED:
            _lib.check(rc, "tbik_gemm_silu_mul_bf16")
        _decline(("silu_tree", M, N, K, leaf_k))
    if (gate.dim() == 2 and up.shape == gate.shape and gate.stride(1) == 1 and up.stride(1) == 1 and gate.stride(0) == up.stride(0)
            and gate.dtype == up.dtype and up.data_ptr() == gate.data_ptr() + K * gate.element_size()
            and (M == 1 or gate.stride(0) >= 2 * K)):
        # the two halves of one merged projection, side by side in memory: the activation kernel reads them in place
        merged = torch.as_strided(gate, (M, 2 * K), (gate.stride(0), 1))
    else:
        merged = torch.cat((gate, up), dim=-1)
    return gemm_tree(bi_silu_mul(merged), B, bias, leaf_k)


def gemm_silu_mul(x: torch.Tensor, W: torch.Tensor) -> torch.Tensor:
    """bi_silu_mul(bi_gemm(x, W.t())) for the merged gate/up weight W [2*inter, K] (nn.Linear layout): one launch
    (`bi_gemm_silu_mul_bf16`) for 5 .. 64 bf16 rows and for the many that run on its 256-row tiles, the two calls
    otherwise.  Same bits either way."""
    _require_gpu(x, W)
    M, K = x.shape
    inter = W.shape[0] // 2
    ldw = W.stride(0)
    fusable = (x.dtype == torch.bfloat16 and W.dtype == torch.bfloat16 and M > 4 and W.shape[0] == 2 * inter and inter % 16 == 0
               and K % 32 == 0 and W.stride(1) == 1 and ldw >= K and ldw % 8 == 0 and _aligned16(W)
               and (M <= 64 or (ldw < _FAR_ROWS and x.stride(0) < _FAR_ROWS))
               and not torch.compiler.is_compiling() and ("mm_silu", M, inter, K) not in _declined)
    if fusable:
        x2, ldx = _rows16(x)
        out = torch.empty((M, inter), device=x.device, dtype=x.dtype)
        rc = _lib.lib().bi_gemm_silu_mul_bf16(x2.data_ptr(), ldx, W.data_ptr(), ldw, out.data_ptr(), out.stride(0), M, inter, K,
                                              _stream(x))
        if rc == _lib.TBIK_OK:
            return out
        if rc != _lib.TBIK_ERR_UNSUPPORTED:
            _lib.check(rc, "bi_gemm_silu_mul_bf16")
        _decline(("mm_silu", M, inter, K))
    return bi_silu_mul(bi_gemm(x, W.t(), None))


# --------------------------------------------------------------------------------------------
# the (add-)RMSNorm behind a row-split layer, inside the launch that combines the layer's K shards
# --------------------------------------------------------------------------------------------
def _norm_after(y: torch.Tensor, residual: Optional[torch.Tensor], norm_weight: Optional[torch.Tensor], eps: float):
    """The two-call form: (bi_rmsnorm(y [+ residual]), new residual or None)."""
    if residual is None:
        return bi_rmsnorm(y, norm_weight, eps), None
    out, res = bi_add_rmsnorm(y, residual, norm_weight, eps)
    return out, res


def gemm_tree_add_rmsnorm(A: torch.Tensor, B: torch.Tensor, bias: Optional[torch.Tensor], leaf_k: int,
                          residual: Optional[torch.Tensor], norm_weight: Optional[torch.Tensor], eps: float):
    """(rms_norm(gemm_tree(A, B, bias, leaf_k) [+ residual]) * norm_weight, new residual or None).

    One call (`tbik_gemm_rmsnorm_bf16`: the norm runs in the launch that combines the matmul's K shards) where the matmul
    of this shape ends in such a combine -- decode- and prefill-sized batches of a row-split layer; the matmul followed
    by the norm otherwise.  Same bits either way."""
    _require_gpu(A, B, bias, residual, norm_weight)
    M, K = A.shape
    N = B.shape[1]
    fusable = (A.dtype == torch.bfloat16 and B.dtype == torch.bfloat16 and M > 0 and N % 8 == 0 and N <= 8192 and B.stride(0) == 1
               and (residual is None or (residual.dtype == torch.bfloat16 and tuple(residual.shape) == (M, N)))
               and (norm_weight is None or norm_weight.dtype == torch.bfloat16) and (bias is None or bias.dtype == torch.bfloat16)
               and not torch.compiler.is_compiling() and ("tree_norm", M, N, K, leaf_k) not in _declined)
    if fusable:
        a, lda = _rows16(A)
        w, ldb_k, ldb_n = _tree_operand(B, M, leaf_k)
        if ldb_k == 1:
            L = _lib.lib()
            b = None if bias is None else bias.contiguous()
            nw = None if norm_weight is None else norm_weight.contiguous()
            r2, ldr = (None, 0) if residual is None else _rows16(residual)
            out = torch.empty((M, N), device=A.device, dtype=A.dtype)
            rout = None if residual is None else torch.empty_like(out)
            ws_bytes = L.tbik_gemm_workspace_bytes(M, N, K, leaf_k)
            ws = torch.empty(ws_bytes, device=A.device, dtype=torch.uint8) if ws_bytes else None
            rc = L.tbik_gemm_rmsnorm_bf16(a.data_ptr(), lda, w.data_ptr(), ldb_k, ldb_n, M, N, K, leaf_k,
                                          None if b is None else b.data_ptr(), None if r2 is None else r2.data_ptr(), ldr,
                                          None if nw is None else nw.data_ptr(), eps,
                                          None if rout is None else rout.data_ptr(), 0 if rout is None else rout.stride(0),
                                          out.data_ptr(), out.stride(0), None if ws is None else ws.data_ptr(), ws_bytes, _stream(A))
            if rc == _lib.TBIK_OK:
                return out, rout
            if rc != _lib.TBIK_ERR_UNSUPPORTED:
                _lib.check(rc, "tbik_gemm_rmsnorm_bf16")
            _decline(("tree_norm", M, N, K, leaf_k))
    return _norm_after(gemm_tree(A, B, bias, leaf_k), residual, norm_weight, eps)


def tree_combine_add_rmsnorm(parts: List[torch.Tensor], bias: Optional[torch.Tensor], residual: Optional[torch.Tensor],
                             norm_weight: Optional[torch.Tensor], eps: float):
    """(rms_norm(tree_combine(parts) (+ bias) [+ residual]) * norm_weight, new residual or None) for 2-D partials: one
    launch (`tbik_tree_combine_rmsnorm_bf16`) for bf16 rows of at most 8192 elements, the separate calls otherwise."""
    _require_gpu(*parts, bias, residual, norm_weight)
    p0 = parts[0]
    n = len(parts)
    fusable = (p0.dim() == 2 and n >= 2 and n <= 32 and (n & (n - 1)) == 0 and all(p.dtype == torch.bfloat16 and p.shape == p0.shape for p in parts)
               and p0.shape[0] > 0 and p0.shape[1] % 8 == 0 and p0.shape[1] <= 8192
               and (residual is None or (residual.dtype == torch.bfloat16 and residual.shape == p0.shape))
               and (norm_weight is None or norm_weight.dtype == torch.bfloat16) and (bias is None or bias.dtype == torch.bfloat16)
               and not torch.compiler.is_compiling())
    if fusable:
        ps = [p.contiguous() for p in parts]
        if all(_aligned16(p) for p in ps):
            M, N = p0.shape
            arr = (ctypes.c_void_p * n)(*[p.data_ptr() for p in ps])
            b = None if bias is None else bias.contiguous()
            nw = None if norm_weight is None else norm_weight.contiguous()
            r2, ldr = (None, 0) if residual is None else _rows16(residual)
            out = torch.empty((M, N), device=p0.device, dtype=p0.dtype)
            rout = None if residual is None else torch.empty_like(out)
            rc = _lib.lib().tbik_tree_combine_rmsnorm_bf16(arr, n, M, N, None if b is None else b.data_ptr(),
                                                           None if r2 is None else r2.data_ptr(), ldr,
                                                           None if nw is None else nw.data_ptr(), eps,
                                                           None if rout is None else rout.data_ptr(), 0 if rout is None else rout.stride(0),
                                                           out.data_ptr(), out.stride(0), _stream(p0))
            _lib.check(rc, "tbik_tree_combine_rmsnorm_bf16")
            return out, rout
    y = parts[0] if n == 1 else tree_combine(parts)
    if bias is not None:
        y = y + bias
    return _norm_after(y, residual, norm_weight, eps)


# --------------------------------------------------------------------------------------------
# q/k norm + rotary embedding + KV-cache write in front of the attention
# --------------------------------------------------------------------------------------------
def bi_qk_norm_rope_cache_bf16(qkv: torch.Tensor, q_weight: torch.Tensor, k_weight: torch.Tensor, inv_freq: torch.Tensor,
                               positions: torch.Tensor, seq_of_token: torch.Tensor, k_cache: torch.Tensor,
                               vt_cache: torch.Tensor, q_heads: int, kv_heads: int, eps: float) -> torch.Tensor:
    """Writes this step's keys and values into the caches (in place) and returns the normed, rotated queries
    [tokens, q_heads, 128]."""
    _require_gpu(qkv, q_weight, k_weight, inv_freq, positions, seq_of_token, k_cache, vt_cache)
    tokens = qkv.shape[0]
    assert qkv.dtype == torch.bfloat16 and qkv.stride(1) == 1 and qkv.shape[1] == (q_heads + 2 * kv_heads) * 128
    assert k_cache.is_contiguous() and vt_cache.is_contiguous() and k_cache.shape[1] == kv_heads and k_cache.shape[3] == 128
    assert positions.dtype == torch.int64 and seq_of_token.dtype == torch.int64 and inv_freq.dtype == torch.float32
    assert positions.numel() == tokens and seq_of_token.numel() == tokens and inv_freq.numel() == 64
    q_out = torch.empty((tokens, q_heads, 128), device=qkv.device, dtype=torch.bfloat16)
    rc = _lib.lib().bi_qk_norm_rope_cache_bf16(
        qkv.data_ptr(), qkv.stride(0), q_weight.contiguous().data_ptr(), k_weight.contiguous().data_ptr(),
        inv_freq.contiguous().data_ptr(), positions.contiguous().data_ptr(), seq_of_token.contiguous().data_ptr(),
        q_out.data_ptr(), k_cache.data_ptr(), vt_cache.data_ptr(), tokens, q_heads, kv_heads, 128,
        k_cache.shape[2], k_cache.shape[0], eps, _stream(qkv))
    _lib.check(rc, "bi_qk_norm_rope_cache_bf16")
    return q_out


def bi_attention_decode_qkv(qkv: torch.Tensor, q_weight: torch.Tensor, k_weight: torch.Tensor, inv_freq: torch.Tensor,
                            k_cache: torch.Tensor, vt_cache: torch.Tensor, ctx_len: torch.Tensor, q_heads: int, kv_heads: int,
                            scale: float, eps: float) -> torch.Tensor:
    """A decode step of an attention block for sequences with one new token each (row b of qkv = sequence b's token at
    position ctx_len[b] - 1): per-head q/k norm, rotary embedding, cache write (in place) and attention in one launch
    (`bi_attention_decode_qkv_ws_bf16`), the two calls where that kernel does not apply.  Same bits either way."""
    _require_gpu(qkv, q_weight, k_weight, inv_freq, k_cache, vt_cache, ctx_len)
    B = qkv.shape[0]
    assert qkv.dtype == torch.bfloat16 and qkv.stride(1) == 1 and qkv.shape[1] == (q_heads + 2 * kv_heads) * 128
    assert k_cache.is_contiguous() and vt_cache.is_contiguous() and k_cache.shape[1] == kv_heads and k_cache.shape[3] == 128
    assert ctx_len.dtype == torch.int32 and ctx_len.numel() == B and k_cache.shape[0] == B and inv_freq.dtype == torch.float32
    max_len = k_cache.shape[2]
    if ("attn_qkv", q_heads, kv_heads, max_len % 32) not in _declined:
        out = torch.empty((B, q_heads, 128), device=qkv.device, dtype=qkv.dtype)
        ws, ws_bytes = _attention_workspace(B, 1, q_heads, kv_heads, max_len, qkv.device)
        rc = _lib.lib().bi_attention_decode_qkv_ws_bf16(
            qkv.data_ptr(), qkv.stride(0) if B > 1 else max(qkv.stride(0), qkv.shape[1]), q_weight.contiguous().data_ptr(),
            k_weight.contiguous().data_ptr(), inv_freq.contiguous().data_ptr(), k_cache.data_ptr(), vt_cache.data_ptr(),
            out.data_ptr(), ctx_len.data_ptr(), B, q_heads, kv_heads, 128, max_len, scale, eps,
            None if ws is None else ws.data_ptr(), ws_bytes, _stream(qkv))
        if rc == _lib.TBIK_OK:
            return out
        if rc != _lib.TBIK_ERR_UNSUPPORTED:
            _lib.check(rc, "bi_attention_decode_qkv_ws_bf16")
        _decline(("attn_qkv", q_heads, kv_heads, max_len % 32))
    pos = (ctx_len - 1).to(torch.int64)
    seq = torch.arange(B, device=qkv.device, dtype=torch.int64)
    q = bi_qk_norm_rope_cache_bf16(qkv, q_weight, k_weight, inv_freq, pos, seq, k_cache, vt_cache, q_heads, kv_heads, eps)
    one = torch.ones(B, dtype=torch.int32, device=qkv.device)
    return bi_attention_bf16(q, k_cache, vt_cache, torch.arange(B, dtype=torch.int32, device=qkv.device), one, ctx_len, 1, scale)


def bi_argmax(logits: torch.Tensor) -> torch.Tensor:
    """Index (int64) of the largest element of each row of a 2-D bf16 tensor, ties resolved to the lowest index."""
    _require_gpu(logits)
    if logits.dim() != 2 or logits.dtype != torch.bfloat16:
        raise NotImplementedError("bi_argmax takes a 2-D bfloat16 tensor")
    x = logits if logits.stride(1) == 1 else logits.contiguous()
    out = torch.empty((x.shape[0],), device=x.device, dtype=torch.int64)
    rc = _lib.lib().bi_argmax_bf16(x.data_ptr(), x.stride(0) if x.shape[0] > 1 else max(x.stride(0), x.shape[1]), out.data_ptr(), x.shape[0], x.shape[1], _stream(x))
    _lib.check(rc, "bi_argmax_bf16")
    return out


def bi_argmax_advance(logits: torch.Tensor, next_token: torch.Tensor, history: Optional[torch.Tensor] = None,
                      count: Optional[torch.Tensor] = None, positions: Optional[torch.Tensor] = None,
                      ctx_len: Optional[torch.Tensor] = None) -> torch.Tensor:
    """bi_argmax written into `next_token` (int64 [rows]) plus the bookkeeping of a decode step in the same launch:
    the index also goes to history[r, count[r]] (int64 [rows, T]; skipped once count[r] reaches T), then count[r]
    (int64), positions[r] (int64) and ctx_len[r] (int32) advance by one.  All tensors are updated in place."""
    _require_gpu(logits)
    if logits.dim() != 2 or logits.dtype != torch.bfloat16:
        raise NotImplementedError("bi_argmax_advance takes a 2-D bfloat16 tensor")
    x = logits if logits.stride(1) == 1 else logits.contiguous()
    rows = x.shape[0]

    def arg(t, dtype, shape, name):
        if t is None:
            return 0
        if t.dtype != dtype or tuple(t.shape) != shape or not t.is_contiguous() or t.device != x.device:
            raise ValueError(f"{name}: a contiguous {dtype} tensor of shape {shape} on {x.device} is required")
        return t.data_ptr()

    if history is not None and (history.dim() != 2 or count is None):
        raise ValueError("history is [rows, T] and needs count")
    T = history.shape[1] if history is not None else 0
    rc = _lib.lib().bi_argmax_advance_bf16(
        x.data_ptr(), x.stride(0) if rows > 1 else max(x.stride(0), x.shape[1]),
        arg(next_token, torch.int64, (rows,), "next_token"), rows, x.shape[1],
        arg(history, torch.int64, (rows, T), "history"), T, arg(count, torch.int64, (rows,), "count"),
        arg(positions, torch.int64, (rows,), "positions"), arg(ctx_len, torch.int32, (rows,), "ctx_len"), _stream(x))
    _lib.check(rc, "bi_argmax_advance_bf16")
    return next_token
