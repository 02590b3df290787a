"""The tree matmul of decode batches (up to 64 rows, weights through a deep LDS ring): against the oracle and against the
rows of a batch that the 128-row tiles serve, bit for bit."""
import pytest
import torch

from llm_reproducibility_amd.tbik import matmul_tp_persistent
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,N,K,leaf", [
    (5, 40, 512, 256),       # two waves, one shard, a tile that is mostly past the edge
    (16, 3071, 2048, 256),   # three waves, an odd last column
    (17, 4093, 2048, 256),   # four
    (32, 5120, 2048, 128),   # five, leaves of two slices
    (33, 5117, 2048, 256),   # five do not divide the 64 rows
    (64, 6143, 2048, 256),   # six
    (49, 24570, 512, 256),   # no cut of K, a level of the tree inside the shard
    (48, 300, 3200, 128),    # groups of 25 leaves, fewer slices in the ring than in the shard
    (20, 1000, 256, 256),    # one leaf: fewer slices than the ring holds
    (33, 300, 1024, 256),    # K in two rather than uncut
])
def test_oracle_and_larger_batch(dev, M, N, K, leaf, f16):
    print("case few", M, N, K, leaf, f16, flush=True)
    dt = torch.float16 if f16 else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(M + N)
    if not f16 and M * N * K < 4e8:
        A, W = O.integer_bf16((M, K), -9, 9, 1), O.integer_bf16((N, K), -7, 7, 2)
        assert torch.equal(matmul_tp_persistent(A.to(dev), W.to(dev).t(), leaf_k=leaf).cpu(), O.matmul_tree(A, W.t(), leaf=leaf))
    x = torch.randn((300, K), generator=gen, device=dev).to(dt)
    w = (torch.randn((N, K), generator=gen, device=dev) * 0.02).to(dt)
    bias = torch.randn(N, generator=gen, device=dev).to(dt)
    for b in (None, bias):
        big = matmul_tp_persistent(x, w.t(), b, leaf_k=leaf)
        assert torch.equal(matmul_tp_persistent(x[:M], w.t(), b, leaf_k=leaf), big[:M])
    padded = torch.zeros((M, K + 8), device=dev, dtype=dt)      # rows with a stride of their own
    padded[:, :K] = x[:M]
    assert torch.equal(matmul_tp_persistent(padded[:, :K], w.t(), leaf_k=leaf), matmul_tp_persistent(x, w.t(), leaf_k=leaf)[:M])


@pytest.mark.parametrize("N,K", [(16384, 4096), (8192, 16384)])
def test_three_levels_inside_a_shard(dev, N, K):
    gen = torch.Generator(device=dev).manual_seed(N)
    x = torch.randn((300, K), generator=gen, device=dev).bfloat16()
    w = (torch.randn((N, K), generator=gen, device=dev) * 0.02).bfloat16()
    big = matmul_tp_persistent(x, w.t())
    for M in (6, 25, 61):
        print("case few levels", M, N, K, flush=True)
        assert torch.equal(matmul_tp_persistent(x[:M], w.t()), big[:M])


# both sides of the size from which on the weights are loaded with the non-temporal hint (64 MB), which the last rows of a matrix do too
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("leaf", [128, 256])
@pytest.mark.parametrize("N", [3906, 3907])
def test_weights_around_the_size_of_the_hint(dev, N, leaf, f16):
    print("case few hint", N, leaf, f16, flush=True)
    dt, K = torch.float16 if f16 else torch.bfloat16, 8192
    gen = torch.Generator(device=dev).manual_seed(N)
    x = torch.randn((300, K), generator=gen, device=dev).to(dt)
    w = (torch.randn((N, K), generator=gen, device=dev) * 0.02).to(dt)
    big = matmul_tp_persistent(x, w.t(), leaf_k=leaf)
    for M in (5, 16, 17, 32, 33, 64):
        assert torch.equal(matmul_tp_persistent(x[:M], w.t(), leaf_k=leaf), big[:M])
