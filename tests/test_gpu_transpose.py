"""The transposing copy and the matmuls that take an operand the other way round through it."""
import pytest
import torch

from llm_reproducibility_amd import ops
from llm_reproducibility_amd.bio import batch_invariant_ops as bio
from llm_reproducibility_amd.tbik import matmul_tp_persistent
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,C,extra", [(2, 2, 0), (64, 64, 0), (65, 63, 8), (31, 257, 56), (333, 72, 0), (1000, 1001, 24), (257, 4096, 8)])
def test_transposing_copy(dev, dtype, R, C, extra):
    """Edges of the 64x64 / 32x32 tiles, columns that allow no 16-byte loads, rows extended by zeros, a column slice."""
    print("case transpose", dtype, R, C, extra, flush=True)
    x = torch.randn((R, C), generator=torch.Generator().manual_seed(R + C)).to(dtype).to(dev)
    k = (R + 7) // 8 * 8 + extra
    out, ld = ops._transposed(x.t(), k)
    assert ld == k and torch.equal(out[:, :R], x.t()) and not out[:, R:].any()
    if C > 16:
        part = x[:, 3:C - 5]
        out, _ = ops._transposed(part.t(), k)
        assert torch.equal(out[:, :R], part.t())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("tokens", [64, 100, 333])
def test_linear_backward_operands(dev, dtype, tokens):
    """Both gradients of a linear layer: the weight as a row-major right operand, the transposed gradient of the output
    against row-major activations with K = tokens of any length.  Integers: every sum is exact (|sum| < 2^11 times a
    power of two or below 2^24), so the result is the exact one rounded once."""
    print("case backward", dtype, tokens, flush=True)
    x = O.integer_bf16((tokens, 264), -3, 3, 1).to(dtype).to(dev)
    w = O.integer_bf16((136, 264), -3, 3, 2).to(dtype).to(dev)
    g = O.integer_bf16((tokens, 136), -2, 2, 3).to(dtype).to(dev)
    gx = (g.double() @ w.double()).to(dtype)
    gw = (g.double().t() @ x.double()).to(dtype)
    assert torch.equal(bio.matmul_persistent(g, w), gx)
    assert torch.equal(bio.matmul_persistent(g.t(), x), gw)
    assert torch.equal(bio.matmul_persistent(g.t()[:1], x), gw[:1])


@pytest.mark.parametrize("K,N", [(2048, 1536), (4096, 2048)])
def test_repacked_and_in_place_agree_around_the_rule(dev, K, N):
    B = O.gaussian_bf16((K, N), 0.02, 3).to(dev)
    Wt = B.t().contiguous().t()
    last = max(128, (ops._TREE_IN_PLACE_MACS - 1) // (K * N))
    for M, tree, in_place in ((last, True, True), (last + 1, True, False), (1, False, False)):
        print("case rule", K, N, M, tree, flush=True)
        A = O.gaussian_bf16((M, K), 1.0, M).to(dev)
        assert (ops._weight_operand(B, M, tree)[1] != 1) == in_place
        f = matmul_tp_persistent if tree else bio.matmul_persistent
        assert torch.equal(f(A, B), f(A, Wt))
