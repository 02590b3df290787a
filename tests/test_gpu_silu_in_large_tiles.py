"""SiLU * up inside the merged gate/up projection on the 256-row tiles against the two calls: same bits."""
import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from llm_reproducibility_amd.bio import batch_invariant_ops as bio

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,inter", [
    (3000, 1024, 2064),   # 256 x 256 tiles: a last tile of 16 columns, a last row tile of 184
    (1025, 256, 4096),    # 256 x 192: one row in the last tile, no whole number of 96 columns, fewer slices than the ring
    (1500, 1024, 4096),   # 192 x 256
    (2049, 512, 2064),    # 192 x 192
])
def test_equals_the_two_calls(dev, M, K, inter):
    print("case silu large", M, K, inter, flush=True)
    gen = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn((M, K), generator=gen, device=dev).mul_(3).bfloat16()
    x[1] *= 100                                  # a gate far beyond both ends of silu
    W = (torch.randn((2 * inter, K), generator=gen, device=dev) * 0.05).bfloat16()
    want = ops.bi_silu_mul(bio.matmul_persistent(x, W.t()))
    s = torch.cuda.current_stream().cuda_stream
    for ldo in (inter, inter + 8, inter + 3):    # the last: rows that allow no 16-byte store
        out = torch.zeros((M, ldo), dtype=torch.bfloat16, device=dev)
        rc = _lib.lib().bi_gemm_silu_mul_bf16(x.data_ptr(), K, W.data_ptr(), K, out.data_ptr(), ldo, M, inter, K, s)
        assert rc == _lib.TBIK_OK
        assert torch.equal(out[:, :inter], want) and not out[:, inter:].any()
    assert torch.equal(ops.gemm_silu_mul(x, W), want)
    assert torch.equal(ops.gemm_silu_mul(x[M - 70:], W), want[M - 70:])   # the two calls


def test_strides_decide_for_their_own_call_only(dev):
    """Rows too far apart for the tiles' 32-bit offsets and a weight of one repeated row go to the two calls; neither is
    remembered against the shape."""
    M, K, inter = 1025, 256, 4096
    gen = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    W = (torch.randn((2 * inter, K), generator=gen, device=dev) * 0.05).bfloat16()
    far = torch.empty((M - 1) * (1 << 22) + K, device=dev, dtype=torch.bfloat16).as_strided((M, K), (1 << 22, 1))
    far.copy_(x)
    want = ops.bi_silu_mul(bio.matmul_persistent(x, W.t()))
    assert torch.equal(ops.gemm_silu_mul(far, W), want)
    del far
    same = W[:1].expand(2 * inter, K)
    assert torch.equal(ops.gemm_silu_mul(x, same), ops.bi_silu_mul(bio.matmul_persistent(x, same.contiguous().t())))
    assert ("mm_silu", M, inter, K) not in ops._declined
    assert torch.equal(ops.gemm_silu_mul(x, W), want) and ("mm_silu", M, inter, K) not in ops._declined
