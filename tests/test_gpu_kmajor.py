"""Matmuls on K-major operands read in place (a row-major right operand, and with it the transposed left operand of a weight
gradient): the bits of the same product on K-contiguous copies, at the edges of tiles and slices."""
import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from llm_reproducibility_amd.tbik import matmul_tp_persistent
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu

# widths of 32, 64, 128 and 256 columns are chosen by the grid; columns and rows end inside tiles, chunks and slices
ONE = [(1, 64, 8), (1, 4096, 4096), (16, 4096, 24576), (40, 128, 1000), (127, 192, 264), (129, 256, 40), (300, 1024, 4104),
       (512, 64, 2048), (1024, 4096, 4096), (1000, 320, 6152), (2048, 128, 8192)]
BOTH = [(8, 1, 8), (8, 63, 264), (136, 64, 1000), (264, 65, 4096), (1024, 127, 1032), (2048, 200, 2048), (1000, 129, 40), (4096, 33, 8192)]


def _operand(g, rows, cols, extra=0, dt=torch.bfloat16):
    t = torch.randn(rows, cols + extra, device="cuda", generator=g).to(dt)
    return t[:, :cols]


def _check(A, B, bias, in_place):
    """in_place: the size is one that the library takes so (None: either way)."""
    direct = ops._bi_gemm_kmajor(A, B, bias, A.dtype is torch.float16)
    if in_place is not None:
        assert (direct is not None) == in_place
    want = ops.bi_gemm(A.contiguous(), B.t().contiguous().t(), bias)
    got = ops.bi_gemm(A, B, bias)
    for out in (got, direct):
        if out is not None:
            assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    return want


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", ONE)
@pytest.mark.parametrize("extra", [0, 24])
def test_row_major_right_operand(M, K, N, extra, dt):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    A, B = _operand(g, M, K, extra, dt), _operand(g, K, N, extra, dt)
    bias = _operand(g, 1, N, 0, dt)[0] if extra else None
    want = _check(A, B, bias, True)
    # one rounding to the type (2^-8, 2^-11) of a sum whose own error is at most K rounding steps of 2^-24 of the sum of magnitudes
    ref = A.double() @ B.double() + (0 if bias is None else bias.double())
    mag = A.double().abs() @ B.double().abs()
    assert ((want.double() - ref).abs() <= ref.abs() * 2.0 ** (-11 if dt is torch.float16 else -8) + mag * (K + 1) * 2.0 ** -24).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", BOTH)
@pytest.mark.parametrize("extra", [0, 8])
def test_both_operands_k_major(M, K, N, extra, dt):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    At, B = _operand(g, K, M, extra, dt), _operand(g, K, N, extra, dt)
    _check(At.t(), B, None, None if K == 1 else True)
    At[-1, 0], B[-1, -1] = float("inf"), float("nan")    # the last row is what stands in for the rows behind K
    _check(At.t(), B, None, None if K == 1 else True)


def test_what_is_left_to_copies():
    g = torch.Generator(device="cuda").manual_seed(5)
    _check(_operand(g, 64, 72), _operand(g, 72, 64), None, False)          # K no whole number of slices
    _check(_operand(g, 64, 64), _operand(g, 64, 60, 4), None, False)       # columns no whole chunks
    _check(_operand(g, 64, 64), _operand(g, 64, 64, 3), None, False)       # rows not aligned
    _check(_operand(g, 64, 65)[:, 1:], _operand(g, 64, 64), None, False)   # left operand not aligned
    _check(_operand(g, 8, 8192), _operand(g, 8192, 128), None, False)      # a few long chains
    _check(_operand(g, 72, 63).t(), _operand(g, 72, 64), None, False)      # M no whole chunks


@pytest.mark.parametrize("M", [0, 3])
def test_empty(M):
    A = torch.empty(M, 64, device="cuda", dtype=torch.bfloat16)
    for N in (0, 8):
        assert ops.bi_gemm(A, torch.empty(64, N, device="cuda", dtype=torch.bfloat16), None).shape == (M, N)


# shards of one and of two groups of leaves, groups of one and of several leaves, tiles that end in rows and columns
TREE = [(1, 256, 8), (3, 4096, 4096), (16, 12288, 1000), (64, 768, 136), (65, 512, 264), (128, 6144, 2048), (129, 25600, 128),
        (300, 2048, 1032), (1024, 1536, 2048), (1000, 8192, 520), (40, 32768, 64)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N", TREE)
def test_tree_row_major(M, K, N, f16):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    dt = torch.float16 if f16 else torch.bfloat16
    A = torch.randn(M, K + 8, device="cuda", generator=g).to(dt)[:, :K]
    B = (torch.randn(K, N + 16, device="cuda", generator=g) * 0.05).to(dt)[:, :N]
    bias = torch.randn(N, device="cuda", generator=g).to(dt)
    native = B.t().contiguous().t()
    want = matmul_tp_persistent(A, native, leaf_k=256)
    assert torch.equal(matmul_tp_persistent(A, B, leaf_k=256), want)
    assert torch.equal(ops.gemm_tree(A, B, bias, 256), ops.gemm_tree(A, native, bias, 256))
    # in place whatever the rule prefers, and with no scratch at all (tiles that need none, or a refusal)
    L, out = _lib.lib(), torch.empty(M, N, device="cuda", dtype=dt)
    f = L.tbik_gemm_f16 if f16 else L.tbik_gemm_bf16
    for nbytes in (L.tbik_gemm_workspace_bytes_rowmajor_b(M, N, K, 256, int(f16)), 0):
        ws = torch.empty(max(nbytes, 16), device="cuda", dtype=torch.uint8)
        out.zero_()
        rc = f(A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), 1, out.data_ptr(), N, M, N, K, 256, None, ws.data_ptr(), nbytes,
               torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.TBIK_OK or (nbytes == 0 and rc == _lib.TBIK_ERR_WORKSPACE)
        if rc == _lib.TBIK_OK:
            assert torch.equal(out, want)


def test_tree_row_major_against_the_oracle():
    x, w = O.integer_bf16((70, 3072), -9, 9, 0), O.integer_bf16((200, 3072), -7, 7, 1)
    B = w.t().contiguous()
    assert torch.equal(matmul_tp_persistent(x.cuda(), B.cuda(), leaf_k=256).cpu(), O.matmul_tree(x, B, leaf=256))


# one row of tiles of every width, grids of one round and of several (128x256, 256x256 and 192x192 tiles), ends in rows and columns
@pytest.mark.parametrize("M,K,N", [(33, 64, 4096), (64, 4096, 768), (65, 128, 6144), (128, 192, 24576), (129, 256, 1030), (384, 128, 24576),
                                   (1000, 320, 6150), (2048, 64, 8192), (2100, 128, 8190), (4096, 128, 5000)])
def test_fp16_rows_in_blocks(M, K, N):
    """fp16 batches on the large tiles: the bits of 32 rows at a time, which run on another kernel."""
    print("case fp16", M, K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A, W = _operand(g, M, K, 8, torch.float16), _operand(g, N, K, 0, torch.float16)
    bias = _operand(g, 1, N, 0, torch.float16)[0]
    for b in (None, bias):
        want = torch.cat([ops.bi_gemm(A[i:i + 32], W.t(), b) for i in range(0, M, 32)])
        assert torch.equal(ops.bi_gemm(A, W.t(), b), want)
