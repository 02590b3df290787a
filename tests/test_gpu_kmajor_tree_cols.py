"""Tree matmuls on a row-major right operand, read in place on tiles of 64 and 128 columns, leaves of 256 and of 128: the bits of
the same product on the K-contiguous copy."""
import ctypes

import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu

# groups of one leaf and of several, uncut and cut, ends in rows, columns and tiles of 64
CASES = [(256, 1024, 1536, 2048), (256, 16, 1024, 4096), (256, 130, 768, 200), (256, 1000, 1024, 5112), (256, 300, 6144, 1032), (256, 1, 256, 72),
         (128, 1, 128, 8), (128, 8, 6400, 5120), (128, 212, 6400, 520), (128, 129, 3200, 136), (128, 50, 25600, 264), (128, 257, 1152, 72),
         (128, 1000, 6400, 1288), (128, 33, 896, 64), (128, 2100, 256, 4096)]


# shards of one and of two groups of leaves (two: the carry and the binary level of the kernel), a group of two leaves and of
# more, on both widths with both leaves: leaf, M, K, N, columns of a tile, cut, groups in a shard
PLANNED = [(128, 129, 768, 2056, 64, 1, 2), (128, 100, 512, 72, 64, 1, 2), (128, 1, 6144, 5112, 64, 8, 2), (128, 33, 2048, 8184, 128, 4, 2),
           (128, 1, 3072, 8184, 128, 4, 2), (128, 33, 5120, 8184, 128, 4, 2), (128, 1, 2560, 8184, 128, 4, 1), (128, 33, 1536, 8184, 128, 4, 1),
           (256, 129, 1536, 4104, 64, 1, 2), (256, 257, 1024, 1032, 64, 1, 2), (256, 1, 8192, 5112, 64, 8, 2), (256, 33, 4096, 5112, 128, 4, 2),
           (256, 129, 1024, 8200, 128, 1, 2), (256, 1, 6144, 5112, 128, 4, 2), (256, 1, 3072, 4104, 128, 4, 1)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("leaf,M,K,N,cols,split,groups", PLANNED)
def test_each_form_of_the_tiles(leaf, M, K, N, cols, split, groups, f16):
    info = (ctypes.c_int * 5)()
    assert _lib.lib().tbik_gemm_plan_info(M, N, K, leaf, int(f16), 1, info) == _lib.TBIK_OK
    assert (info[2], info[1]) == (cols, split) and _lib.tree_params(K // split, leaf)[2] == groups
    test_row_major_tiles(leaf, M, K, N, f16)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("leaf,M,K,N", CASES)
def test_row_major_tiles(leaf, M, K, N, f16):
    print("case row-major tiles", leaf, M, K, N, f16, flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    dt = torch.float16 if f16 else torch.bfloat16
    A = torch.randn(M, K + 8, device="cuda", generator=g).to(dt)[:, :K]
    B = (torch.randn(K, N + 16, device="cuda", generator=g) * 0.05).to(dt)[:, :N]
    bias = torch.randn(N, device="cuda", generator=g).to(dt)
    native = B.t().contiguous().t()
    want = ops.gemm_tree(A, native, None, leaf)
    assert torch.equal(ops.gemm_tree(A, B, None, leaf), want)
    assert torch.equal(ops.gemm_tree(A, B, bias, leaf), ops.gemm_tree(A, native, bias, leaf))
    # in place whatever the rule prefers, and with no scratch at all (tiles that need none, or a refusal)
    L, out = _lib.lib(), torch.empty(M, N, device="cuda", dtype=dt)
    f = L.tbik_gemm_f16 if f16 else L.tbik_gemm_bf16
    for nbytes in (L.tbik_gemm_workspace_bytes_rowmajor_b(M, N, K, leaf, int(f16)), 0):
        ws = torch.empty(max(nbytes, 16), device="cuda", dtype=torch.uint8)
        out.zero_()
        rc = f(A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), 1, out.data_ptr(), N, M, N, K, leaf, None, ws.data_ptr(), nbytes,
               torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.TBIK_OK or (nbytes == 0 and rc == _lib.TBIK_ERR_WORKSPACE)
        if rc == _lib.TBIK_OK:
            assert torch.equal(out, want)


@pytest.mark.parametrize("leaf,M,K,N", [(128, 1000, 12800, 5120), (256, 2048, 6144, 2048)])
def test_scratch_that_cannot_be_used(leaf, M, K, N):
    """Enough scratch at an odd address, or none with its size: the 64-row tiles, which need none for these shapes."""
    print("case unusable scratch", leaf, M, K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    A, B = torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(K, N, device="cuda", generator=g) * 0.05).bfloat16()
    L, out, want = _lib.lib(), torch.empty(M, N, device="cuda", dtype=torch.bfloat16), ops.gemm_tree(A, B, None, leaf)
    nbytes = L.tbik_gemm_workspace_bytes_rowmajor_b(M, N, K, leaf, 0)
    assert nbytes > 0
    ws = torch.empty(nbytes + 16, device="cuda", dtype=torch.uint8)
    for ptr in (ws.data_ptr() + 8, None):
        out.zero_()
        assert L.tbik_gemm_bf16(A.data_ptr(), K, B.data_ptr(), N, 1, out.data_ptr(), N, M, N, K, leaf, None, ptr, nbytes,
                                torch.cuda.current_stream().cuda_stream) == _lib.TBIK_OK
        assert torch.equal(out, want)


def test_leaves_of_128_against_the_oracle():
    x, w = O.integer_bf16((70, 3200), -9, 9, 0), O.integer_bf16((200, 3200), -7, 7, 1)
    B = w.t().contiguous()
    assert torch.equal(ops.gemm_tree(x.cuda(), B.cuda(), None, 128).cpu(), O.matmul_tree(x, B, leaf=128))
