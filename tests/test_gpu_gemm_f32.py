"""fp32 matmuls at the edges of the kernel's tiles.  The operands are small integers, so every product and every partial
sum is exact in fp32 (|sum| <= 63 * K < 2^24) and any order of additions gives the same bits: equality, no tolerance."""
import pytest
import torch

from llm_reproducibility_amd.bio import batch_invariant_ops as bio
from llm_reproducibility_amd.tbik import matmul_tp_persistent
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu

# M, N, K: one row, one k chunk, K ending inside a slice of 32, remainders in every direction, and grids that bring each
# tile (32x32, 64x32, 64x64, 128x128) into use
MM = [(1, 1, 16), (5, 33, 48), (17, 130, 16), (31, 4096, 80), (65, 6150, 48), (190, 4100, 272), (520, 6140, 64),
      (1000, 4090, 48), (1025, 6145, 112)]
TREE = [(1, 3, 128), (33, 65, 128), (16, 4100, 384), (70, 6150, 640), (257, 4090, 1024), (130, 514, 3200)]


def _operands(M, N, K, dev):
    x = O.integer_bf16((M, K), -9, 9, 8 + M).float()
    w = O.integer_bf16((N, K), -7, 7, 9 + N).float()
    return x, w, x.to(dev), w.to(dev)


@pytest.mark.parametrize("M,N,K", MM)
def test_fp32_mm_tile_edges(dev, M, N, K):
    print("case fp32 mm", M, N, K, flush=True)
    x, w, xd, wd = _operands(M, N, K, dev)
    bias = torch.arange(N, dtype=torch.float32) - N // 2
    want = x @ w.t()
    assert torch.equal(bio.matmul_persistent(xd, wd.t()).cpu(), want)
    assert torch.equal(bio.matmul_persistent(xd, wd.t(), bias.to(dev)).cpu(), want + bias)
    wide = torch.full((M, K + 20), float("nan"), device=dev)          # a column slice of a wider tensor, in place
    wide[:, 4:K + 4] = xd
    assert torch.equal(bio.matmul_persistent(wide[:, 4:K + 4], wd.t()).cpu(), want)


@pytest.mark.parametrize("M,N,K", TREE)
def test_fp32_tree_tile_edges(dev, M, N, K):
    print("case fp32 tree", M, N, K, flush=True)
    x, w, xd, wd = _operands(M, N, K, dev)
    assert torch.equal(matmul_tp_persistent(xd, wd.t()).cpu(), x @ w.t())
    # non-integer operands: a row has the bits it has alone, whichever tile serves the batch
    xr, wr = xd + 0.37 * xd.sin(), wd * 0.13
    full = matmul_tp_persistent(xr, wr.t())
    assert torch.equal(matmul_tp_persistent(xr[-1:], wr.t()), full[-1:])


def test_fp32_rows_far_apart(dev):
    """Operand rows so far apart that a tile of 32 does not reach them all with 32-bit byte offsets."""
    M, N, K, ld = 40, 33, 128, 36_000_000
    x, w, xd, wd = _operands(M, N, K, dev)
    far = torch.empty((M - 1) * ld + K, device=dev).as_strided((M, K), (ld, 1))
    far.copy_(xd)
    assert torch.equal(bio.matmul_persistent(far, wd.t()).cpu(), x @ w.t())
    assert torch.equal(matmul_tp_persistent(wd, far.t()).cpu(), w @ x.t())
    assert torch.equal(bio.matmul_persistent(far[:3], wd.t()).cpu(), (x @ w.t())[:3])
