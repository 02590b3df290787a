"""Decode batches on wide matrices: every group width of the ring kernel gives the bits of the product in column chunks."""
import pytest
import torch

from llm_reproducibility_amd import ops

pytestmark = pytest.mark.gpu


# 16-column strips around the lines of the rule (512, 768, 1024, 1536) and a last strip that ends early; K of one slice, below and
# at the lines of the rule, and with the ring not filled; rows around the blocks of 16
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("N", [8192, 8200, 12288, 12296, 16384, 16392, 24576, 24584])
@pytest.mark.parametrize("K", [128, 1024, 4096])
def test_wide_matrix_in_chunks(N, K, f16):
    print("case wide", N, K, f16, flush=True)
    g = torch.Generator(device="cuda").manual_seed(N + K)
    dt = torch.float16 if f16 else torch.bfloat16
    W = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(dt)
    for M in (5, 16, 17, 33, 64):
        x = torch.randn(M, K, device="cuda", generator=g).to(dt)
        got = ops.bi_gemm(x, W.t(), None)
        want = torch.cat([ops.bi_gemm(x, W[i:i + 2048].t(), None) for i in range(0, N, 2048)], dim=1)
        assert torch.equal(got, want)
    ref, mag = x.double() @ W.double().t(), x.double().abs() @ W.double().abs().t()
    # one rounding to the type (2^-8, 2^-11) of a sum whose own error is at most K rounding steps of 2^-24 of the magnitudes
    assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** (-11 if f16 else -8) + mag * (K + 1) * 2.0 ** -24).all()


# both halves of a merged projection on one, two, three and four waves
@pytest.mark.parametrize("inter", [16, 4096, 8192, 12288, 16400])
@pytest.mark.parametrize("K", [512, 4096])
def test_gated_widths(inter, K):
    print("case gated", inter, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(inter + K)
    W = (torch.randn(2 * inter, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    for M in (5, 16, 17, 48, 64):
        x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
        both = torch.cat([ops.bi_gemm(x, W[i:i + 1024].t(), None) for i in range(0, 2 * inter, 1024)], dim=1)
        assert torch.equal(ops.gemm_silu_mul(x, W), ops.bi_silu_mul(both))


# a short K that the ring kernel leaves on very wide matrices: both sides of the rows, the columns and the fill of the rounds from which on
# all of X is staged at once, a last group that ends early
@pytest.mark.parametrize("N", [65536, 65552, 81920, 100000, 128255])
@pytest.mark.parametrize("K", [512, 896])
def test_short_k_of_a_very_wide_matrix(N, K):
    print("case short k", N, K, flush=True)
    g = torch.Generator(device="cuda").manual_seed(N + K)
    W = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(torch.bfloat16)
    for M in (3, 8, 9):
        x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
        got = ops.bi_gemm(x, W.t(), None)
        want = torch.cat([ops.bi_gemm(x, W[i:i + 2048].t(), None) for i in range(0, N, 2048)], dim=1)
        assert torch.equal(got, want)
