"""The forms of the decode attention kernel (two or three slots of value-tile pairs, the chunks walked by one work-group or shared)
at caches that end in the middle of a pair: the bits of the one-wave kernel, and of the step that is made of two launches."""
import ctypes
import math

import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu
D, SCALE = 128, 1.0 / math.sqrt(128)

# query heads, KV heads, sequences, cache length, work-groups per (sequence, KV head), slots of pairs
FORMS = [
    (32, 8, 4, 160, 1, 3), (8, 2, 3, 1056, 3, 3), (16, 8, 2, 2592, 6, 3),       # up to 256 work-groups
    (32, 8, 33, 160, 1, 2), (8, 8, 41, 224, 1, 2), (64, 8, 64, 96, 1, 2),       # 257 .. 512, a chunk each or all of them
    (32, 8, 8, 2592, 6, 2), (16, 8, 12, 2592, 5, 2), (64, 8, 12, 2624, 5, 2), (8, 8, 12, 1120, 3, 2),
    (32, 8, 65, 160, 1, 3), (64, 8, 66, 96, 1, 3), (8, 8, 70, 1120, 1, 3),      # more
]


def _contexts(B, L, least):
    """One key, around the edges of tiles, of pairs and of chunks, and the ends of the cache."""
    edges = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 129, 511, 512, 513, 545, 1024, 1025, 1057, 1537, 2049, 2561, L - 64, L - 32, L - 31, L - 1, L]
    use = [c for c in edges if least <= c <= L]
    return [L] + [use[(5 * b) % len(use)] for b in range(1, B)]


@pytest.mark.parametrize("hq,hkv,B,L,shared,slots", FORMS)
def test_forms(dev, hq, hkv, B, L, shared, slots):
    print("case decode forms", hq, hkv, B, L, flush=True)
    gen = torch.Generator(device=dev).manual_seed(hq + B + L)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    lib, info = _lib.lib(), (ctypes.c_int * 6)()
    rows = 16 * hkv // hq
    kc, vt = rnd(B, hkv, L, D), rnd(B, hkv, D, L)
    pad = torch.nn.functional.pad
    for new in {1, min(rows, 2), rows}:
        nbytes = lib.bi_attention_workspace_bytes(B, new, hq, hkv, L)
        assert lib.bi_attention_plan_info(B, new, hq, hkv, L, nbytes, info) == _lib.TBIK_OK
        assert list(info)[:4] == [2, shared, slots, rows]
        qlens = [max(1, new - b % 3) for b in range(B)]
        ctxs = [max(n, c) for n, c in zip(qlens, _contexts(B, L, 1))]
        starts = [sum(qlens[:b]) for b in range(B)]
        q = rnd(sum(qlens), hq, D)
        args = (i32(starts), i32(qlens), i32(ctxs), new, SCALE)
        got = ops.bi_attention_bf16(q, kc, vt, *args)
        assert torch.equal(got, ops.bi_attention_bf16(q, pad(kc, (0, 0, 0, 4)), pad(vt, (0, 4)), *args))   # the one-wave kernel
    # the step that forms its own query, key and value: the new key in the first and in the second tile of a pair
    qkv, w, inv = rnd(B, (hq + 2 * hkv) * D), (1 + 0.1 * torch.randn(D, generator=gen, device=dev)).to(torch.bfloat16), O.rope_inv_freq(D, 1e6).to(dev)
    for shift in (0, 3):
        ctxs = _contexts(B, L, 1)
        ctxs = ctxs[shift:] + ctxs[:shift]
        ctx = i32(ctxs)
        k1, v1, k2, v2 = kc.clone(), vt.clone(), kc.clone(), vt.clone()
        q = ops.bi_qk_norm_rope_cache_bf16(qkv, w, w, inv, ctx.long() - 1, torch.arange(B, device=dev), k1, v1, hq, hkv, 1e-6)
        want = ops.bi_attention_bf16(q, pad(k1, (0, 0, 0, 4)), pad(v1, (0, 4)), i32(list(range(B))), i32([1] * B), ctx, 1, SCALE)
        got = ops.bi_attention_decode_qkv(qkv, w, w, inv, k2, v2, ctx, hq, hkv, SCALE, 1e-6)
        assert torch.equal(got, want) and torch.equal(k1, k2) and torch.equal(v1, v2)
