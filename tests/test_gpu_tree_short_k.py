"""The tree matmul of short K shards on 128 x 128 tiles: a product of the whole batch against the same rows in small batches
(which other kernels serve) and, where that is quick, against the oracle, bit for bit."""
import ctypes

import pytest
import torch

from llm_reproducibility_amd import _lib
from llm_reproducibility_amd.tbik import matmul_tp_persistent
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (65, 6140, 1024),    # one row of tiles, half empty; the last column tile ragged, stores element by element at its end
    (129, 8190, 512),    # a second row of tiles with one row, two leaves
    (384, 4096, 768),    # 96 work-groups: uncut, three leaves in a group
    (1000, 4093, 1536),  # 256: six leaves, two groups; odd columns
    (1024, 2048, 1536),  # cut in two
    (300, 2049, 3072),   # cut in four, a last tile of one column
    (2041, 2048, 1024),  # sixteen rows of tiles
])
def test_equals_small_batches(dev, M, N, K, f16):
    print("case short k", M, N, K, f16, flush=True)
    info = (ctypes.c_int * 5)()
    assert _lib.lib().tbik_gemm_plan_info(M, N, K, 256, int(f16), 0, info) == _lib.TBIK_OK
    assert info[0] == 1
    dt = torch.float16 if f16 else torch.bfloat16
    gen = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device=dev).to(dt)
    w = (torch.randn((N, K), generator=gen, device=dev) * 0.02).to(dt)
    bias = torch.randn(N, generator=gen, device=dev).to(dt)
    for b in (None, bias):
        got = matmul_tp_persistent(x, w.t(), b)
        for lo in (0, M // 2, M - 49):
            assert torch.equal(matmul_tp_persistent(x[lo:lo + 49], w.t(), b), got[lo:lo + 49])
    if not f16 and M * N * K < 7e8:
        A, W = O.integer_bf16((M, K), -9, 9, 1), O.integer_bf16((N, K), -7, 7, 2)
        assert torch.equal(matmul_tp_persistent(A.to(dev), W.to(dev).t()).cpu(), O.matmul_tree(A, W.t()))


def test_rows_far_apart(dev):
    M, N, K, ld = 384, 4096, 512, 1 << 22
    gen = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    w = torch.randn((N, K), generator=gen, device=dev).bfloat16()
    far = torch.empty((M - 1) * ld + K, device=dev, dtype=torch.bfloat16).as_strided((M, K), (ld, 1))
    far.copy_(x)
    assert torch.equal(matmul_tp_persistent(far, w.t()), matmul_tp_persistent(x, w.t()))
