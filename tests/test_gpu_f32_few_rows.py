"""The fp32 tree matmul of few rows (K cut over the waves of a work-group): the bits of the same rows inside a larger batch."""
import pytest
import torch

from llm_reproducibility_amd.tbik import matmul_tp_persistent

pytestmark = pytest.mark.gpu


# groups of one and of several leaves, four to many groups (fewer stay on the tiles, as the 300 rows do: both sides are one kernel there);
# columns that end inside a strip, and both sides of one round of work-groups; a single slice ring turn and many
@pytest.mark.parametrize("K", [256, 512, 1024, 1536, 3072, 12288, 16384])
@pytest.mark.parametrize("N", [8, 40, 2048, 4096, 4099, 5120])
def test_rows_of_a_larger_batch(K, N):
    print("case f32", K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    x = torch.randn(300, K + 4, device="cuda", generator=g)[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g) * 0.05
    bias = torch.randn(N, device="cuda", generator=g)
    # what is compared with runs on the tiles: 300 rows of at least 1024 columns are more than the 512 blocks that the split takes
    wide = torch.cat([w, torch.randn(max(0, 1024 - N), K, device="cuda", generator=g)])
    for b in (None, bias):
        more = None if b is None else torch.cat([b, torch.zeros(wide.shape[0] - N, device="cuda")])
        want = matmul_tp_persistent(x, wide.t(), more, leaf_k=128)[:, :N]
        for M in (1, 15, 16, 17, 32, 33, 64, 65, 128):
            assert torch.equal(matmul_tp_persistent(x[:M], w.t(), b, leaf_k=128), want[:M]), M
    # fp32 sums: at most K + log2(K) roundings of 2^-24 of the sum of magnitudes
    ref, mag = x.double() @ w.double().t() + bias.double(), x.double().abs() @ w.double().abs().t() + bias.double().abs()
    assert ((want.double() - ref).abs() <= mag * (K + 16) * 2.0 ** -24).all()


def test_special_values():
    x = torch.zeros(5, 2048, device="cuda")
    w = torch.ones(32, 2048, device="cuda")
    x[0, 2047], x[1, 0], x[2, 1000], x[3, 5], x[3, 2000] = float("inf"), float("nan"), -1e38, 3e38, 3e38
    out = matmul_tp_persistent(x, w.t(), leaf_k=128)
    assert torch.isinf(out[0]).all() and torch.isnan(out[1]).all() and (out[2] == -1e38).all()
    assert torch.isinf(out[3]).all() and (out[4] == 0).all()
