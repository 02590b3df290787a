"""The ranks of a row-split layer in one grid: the bits of a product per rank and the shard tree."""
import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from llm_reproducibility_amd.tbik import matmul_tp_persistent, tree_combine
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu


# edges of the tiles of every kernel a plan may choose (rows around 16, 64, 128 and 256; columns that are no multiple of four),
# ranks of one leaf and of odd numbers of leaves, both leaf sizes, the most ranks there can be
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N,leaf,tp", [
    (1, 2048, 512, 256, 8), (5, 12288, 300, 256, 8), (16, 3200 * 2, 130, 128, 2), (17, 8192, 1024, 256, 32), (33, 6144, 2048, 256, 4),
    (64, 25600, 640, 128, 8), (65, 4096, 1030, 256, 2), (129, 25600, 512, 128, 4), (200, 6144, 2048, 256, 8), (257, 4096, 4096, 256, 4),
    (700, 12288, 1500, 256, 2), (130, 1024, 258, 128, 8),
])
def test_ranks_in_one_grid(dev, M, K, N, leaf, tp, f16):
    print("case ranks", M, K, N, leaf, tp, f16, flush=True)
    gen = torch.Generator(device=dev).manual_seed(M + N)
    dt = torch.float16 if f16 else torch.bfloat16
    wide = torch.randn((M, K + 8), generator=gen, device=dev).to(dt)
    x, w = wide[:, :K], (torch.randn((N, K), generator=gen, device=dev) * 0.02).to(dt)   # rows further apart than K
    ks = K // tp
    parts = [matmul_tp_persistent(x[:, r * ks:(r + 1) * ks], w[:, r * ks:(r + 1) * ks].t(), leaf_k=leaf) for r in range(tp)]
    assert torch.equal(ops.gemm_tree_sharded(x, w, leaf, tp), tree_combine(parts))


def test_ranks_against_the_oracle(dev):
    x, w = O.integer_bf16((70, 3072), -9, 9, 0), O.integer_bf16((200, 3072), -7, 7, 1)
    want = O.matmul_tree(x, w.t(), leaf=128)
    for tp in (2, 8):
        assert torch.equal(ops.gemm_tree_sharded(x.to(dev), w.to(dev), 128, tp).cpu(), want)


def test_refused(dev):
    x, w = torch.zeros((4, 1536), device=dev, dtype=torch.bfloat16), torch.zeros((64, 1536), device=dev, dtype=torch.bfloat16)
    for leaf, tp in ((256, 3), (256, 4), (256, 64), (64, 2)):     # no power of two, no whole leaves, too many ranks, no such leaf
        with pytest.raises(_lib.TbikError):
            ops.gemm_tree_sharded(x, w, leaf, tp)
    with pytest.raises(NotImplementedError):
        ops.gemm_tree_sharded(x, w.half(), 256, 2)
