"""The single-accumulator matmul of decode batches on the LDS ring: against the rows of a larger batch, which other kernels
serve, bit for bit; the gated form against the two calls."""
import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from llm_reproducibility_amd.bio import batch_invariant_ops as bio

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (5, 40, 128),        # one slice; a last strip of eight columns
    (16, 4095, 640),     # one strip per work-group, fewer slices than the ring holds, odd columns
    (17, 1000, 2048),    # two strips, a second block with one row
    (32, 8191, 256),
    (3, 2047, 4096),
    (31, 10229, 1280),   # three strips
    (9, 65999, 256),     # four strips, many rounds
    (33, 4111, 1408),    # three and four blocks of rows (fp16)
    (64, 24571, 256),    # six strips (fp16)
])
def test_rows_of_a_larger_batch(dev, M, N, K, f16):
    print("case ring", M, N, K, f16, flush=True)
    dt = torch.float16 if f16 else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((200, K), generator=gen, device=dev).to(dt)
    w = (torch.randn((N, K), generator=gen, device=dev) * 0.02).to(dt)
    bias = torch.randn(N, generator=gen, device=dev).to(dt)
    for b in (None, bias):
        big = bio.matmul_persistent(x, w.t(), b)
        assert torch.equal(bio.matmul_persistent(x[:M], w.t(), b), big[:M])
    wide = torch.full((M, K + 8), float("nan"), device=dev, dtype=dt)      # rows with a stride of their own
    wide[:, :K] = x[:M]
    assert torch.equal(bio.matmul_persistent(wide[:, :K], w.t()), bio.matmul_persistent(x, w.t())[:M])


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("K,inter", [(512, 16), (640, 1552), (1024, 6160), (512, 9728), (2048, 17424)])
def test_gated_equals_the_two_calls(dev, M, K, inter):
    print("case ring gated", M, K, inter, flush=True)
    gen = torch.Generator(device=dev).manual_seed(M + inter)
    x = torch.randn((M, K), generator=gen, device=dev).mul_(3).bfloat16()
    x[1] *= 100
    W = (torch.randn((2 * inter, K), generator=gen, device=dev) * 0.05).bfloat16()
    want = ops.bi_silu_mul(bio.matmul_persistent(x, W.t()))
    assert torch.equal(ops.gemm_silu_mul(x, W), want)
    out = torch.zeros((M, inter + 3), dtype=torch.bfloat16, device=dev)    # rows that allow no 8-byte store
    rc = _lib.lib().bi_gemm_silu_mul_bf16(x.data_ptr(), K, W.data_ptr(), K, out.data_ptr(), inter + 3, M, inter, K,
                                          torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.TBIK_OK
    assert torch.equal(out[:, :inter], want) and not out[:, inter:].any()
