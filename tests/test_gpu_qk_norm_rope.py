"""q/k norm, rotary embedding and cache write at the edges of the kernel's units: 64 tokens and 128, 32 or 8 channels per
value tile, one to eight heads per wavefront, tokens side by side and one for each of many sequences."""
import pytest
import torch

from llm_reproducibility_amd import ops
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,lens,prefix", [(8, 1, [1], 0), (5, 3, [63, 2], 7), (32, 8, [64], 0), (9, 9, [65, 30, 40], 3), (16, 2, [300], 33),
                                                (4, 1, [1] * 70, 5), (8, 8, [1] * 257, 2), (8, 16, [1000], 0), (64, 8, [513], 1)])
def test_units_and_remainders(dev, hq, hkv, lens, prefix):
    print("case qk_norm_rope", hq, hkv, lens, flush=True)
    T, B, L = sum(lens), len(lens), (max(lens) + prefix + 31) // 32 * 32
    qkv = O.gaussian_bf16((T, (hq + 2 * hkv) * 128), 1.0, T).to(dev)
    qw = (1.0 + 0.1 * torch.randn(128, generator=torch.Generator().manual_seed(1))).to(torch.bfloat16).to(dev)
    kw = (1.0 + 0.1 * torch.randn(128, generator=torch.Generator().manual_seed(2))).to(torch.bfloat16).to(dev)
    inv = O.rope_inv_freq(128, 1e6).to(dev)
    pos = torch.cat([torch.arange(prefix, prefix + n) for n in lens]).to(dev)
    seq = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).to(dev)
    fill = 7.0                                                    # every cache entry that is not a token's stays as it was
    kc = torch.full((B, hkv, L, 128), fill, dtype=torch.bfloat16, device=dev)
    vt = torch.full((B, hkv, 128, L), fill, dtype=torch.bfloat16, device=dev)
    q = ops.bi_qk_norm_rope_cache_bf16(qkv, qw, kw, inv, pos, seq, kc, vt, hq, hkv, 1e-6)
    c = qkv.cpu().reshape(T, hq + 2 * hkv, 128)
    want_q = O.qk_norm_rope(c[:, :hq], qw.cpu(), 1e-6, pos.cpu(), inv.cpu())
    want_k = O.qk_norm_rope(c[:, hq:hq + hkv], kw.cpu(), 1e-6, pos.cpu(), inv.cpu())
    assert not O.outside_tolerance(q.cpu(), want_q).any()         # the stated tolerance: 1 bf16 ulp or 2^-8 of the scale
    k_all, v_all = torch.full_like(kc, fill), torch.full_like(vt, fill)
    k_all[seq, :, pos] = kc[seq, :, pos]
    v_all[seq, :, :, pos] = qkv[:, (hq + hkv) * 128:].reshape(T, hkv, 128)
    assert torch.equal(kc, k_all) and torch.equal(vt, v_all)
    assert not O.outside_tolerance(kc[seq, :, pos].cpu(), want_k).any()
    # a token alone, out of range tokens ignored
    kc1, vt1 = kc.clone().fill_(fill), vt.clone().fill_(fill)
    bad = seq.clone()
    bad[: T - 1] = B
    q1 = ops.bi_qk_norm_rope_cache_bf16(qkv, qw, kw, inv, pos, bad, kc1, vt1, hq, hkv, 1e-6)
    assert torch.equal(q1, q)
    s, p = int(seq[-1]), int(pos[-1])
    assert torch.equal(kc1[s, :, p], kc[s, :, p]) and torch.equal(vt1[s, :, :, p], vt[s, :, :, p])
    assert int((kc1 != fill).any(-1).sum()) <= hkv and int((vt1 != fill).any(-1).any(-1).sum()) <= hkv
