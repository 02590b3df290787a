"""Attention around the edges of its 512-key chunks: the kernels that walk all chunks, the ones that share them between
work-groups and the one-wave kernel give the same bits, and the values are those of the float64 oracle."""
import math

import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu
D, SCALE = 128, 1.0 / math.sqrt(128)


def _caches(ks, vs, L, dev):
    kc = torch.zeros((len(ks), ks[0].shape[1], L, D), dtype=torch.bfloat16, device=dev)
    vt = torch.zeros((len(ks), ks[0].shape[1], D, L), dtype=torch.bfloat16, device=dev)
    for b, (k, v) in enumerate(zip(ks, vs)):
        kc[b, :, : k.shape[0]] = k.transpose(0, 1)
        vt[b, :, :, : v.shape[0]] = v.permute(1, 2, 0)
    return kc, vt


def _no_workspace(monkeypatch):
    monkeypatch.setattr(ops, "_attention_workspace", lambda *a: (None, 0))


# heads per KV head 4, 8, 1 (decode rows) and more new queries than a decode tile takes (the grouped kernel); contexts one key
# around one, two and three chunks, and one whose queries straddle an edge
@pytest.mark.parametrize("hq,hkv,new,ctxs", [
    (8, 2, 1, [1, 511, 512, 513, 1023, 1024, 1025, 1537]),
    (16, 2, 2, [513, 514, 1025, 2, 1600]),
    (3, 3, 5, [515, 1027, 1540]),
    (8, 2, 40, [40, 520, 530, 1056, 1560]),
    (2, 2, 20, [1030, 1545]),
])
def test_chunk_edges(dev, monkeypatch, hq, hkv, new, ctxs):
    torch.manual_seed(hq + new)
    print("case chunks", hq, hkv, new, ctxs, flush=True)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    rnd = lambda *s: torch.randn(s, device=dev).to(torch.bfloat16)  # noqa: E731
    ks, vs = [rnd(c, hkv, D) for c in ctxs], [rnd(c, hkv, D) for c in ctxs]
    qlens = [min(new, c) - (b % 2 if min(new, c) > 1 else 0) for b, c in enumerate(ctxs)]      # ragged
    qs = [rnd(n, hq, D) for n in qlens]
    starts = [sum(qlens[:i]) for i in range(len(qlens))]
    args = (i32(starts), i32(qlens), i32(ctxs), new, SCALE)
    L = (max(ctxs) + 31) // 32 * 32
    q = torch.cat(qs)
    assert _lib.lib().bi_attention_workspace_bytes(len(ctxs), new, hq, hkv, L) > 0
    kc, vt = _caches(ks, vs, L, dev)
    shared = ops.bi_attention_bf16(q, kc, vt, *args)
    for b, c in enumerate(ctxs):
        want = O.causal_attention(qs[b].cpu(), ks[b].cpu(), vs[b].cpu(), SCALE).to(torch.bfloat16)
        assert not O.outside_tolerance(shared[starts[b]: starts[b] + qlens[b]].cpu(), want).any(), c
    kc2, vt2 = _caches(ks, vs, L + 4, dev)                      # no whole number of tiles: the one-wave kernel
    assert torch.equal(ops.bi_attention_bf16(q, kc2, vt2, *args), shared)
    kc3, vt3 = _caches(ks, vs, L + 4096, dev)                   # a longer cache: another number of chunks and work-groups
    assert torch.equal(ops.bi_attention_bf16(q, kc3, vt3, *args), shared)
    for b in (0, len(ctxs) - 1):                                # a sequence alone
        kb, vb = _caches([ks[b]], [vs[b]], (ctxs[b] + 31) // 32 * 32, dev)
        alone = ops.bi_attention_bf16(qs[b], kb, vb, i32([0]), i32([qlens[b]]), i32([ctxs[b]]), qlens[b], SCALE)
        assert torch.equal(alone, shared[starts[b]: starts[b] + qlens[b]])
    _no_workspace(monkeypatch)
    assert torch.equal(ops.bi_attention_bf16(q, kc, vt, *args), shared)


# one launch of each form that the grouped kernel takes once the chip is full (query heads, KV heads, sequences, longest
# number of new tokens): two blocks of queries per work-group, eight heads, one block, and eight heads of a few queries
@pytest.mark.parametrize("hq,hkv,B,new", [(32, 8, 20, 80), (16, 8, 26, 80), (16, 16, 17, 80), (64, 8, 13, 80), (32, 8, 16, 80), (64, 8, 65, 8)])
def test_forms_for_a_full_chip(dev, hq, hkv, B, new):
    """Ragged prompts and chunks around the edges of blocks of 16 and 32 queries, of tiles and of chunks: the bits of the
    one-wave kernel, and of a sequence alone in a short cache."""
    print("case full chip", hq, hkv, B, new, flush=True)
    gen = torch.Generator(device=dev).manual_seed(hq + B)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    qlens = [min(new, (80, 1, 17, 32, 33, 79, 16, 49)[b % 8]) for b in range(B)]
    ctxs = [max(n, (1100, 512, 513, 80, 1024, 1025, 530, 545, 1056)[b % 9]) for b, n in enumerate(qlens)]
    L = 1120
    assert ((new + 15) // 16) * hkv * B > 512                   # beyond the forms with loader waves
    starts = [sum(qlens[:i]) for i in range(B)]
    q, kc, vt = rnd(sum(qlens), hq, D), rnd(B, hkv, L, D), rnd(B, hkv, D, L)
    args = (i32(starts), i32(qlens), i32(ctxs), new, SCALE)
    got = ops.bi_attention_bf16(q, kc, vt, *args)
    pad = torch.nn.functional.pad
    assert torch.equal(ops.bi_attention_bf16(q, pad(kc, (0, 0, 0, 4)), pad(vt, (0, 4)), *args), got)   # the one-wave kernel
    for b in (0, 5, B - 1):
        n, short = qlens[b], (ctxs[b] + 31) // 32 * 32
        alone = ops.bi_attention_bf16(q[starts[b]: starts[b] + n], kc[b: b + 1, :, :short].contiguous(), vt[b: b + 1, :, :, :short].contiguous(),
                                      i32([0]), i32([n]), i32([ctxs[b]]), n, SCALE)
        assert torch.equal(alone, got[starts[b]: starts[b] + n])


@pytest.mark.parametrize("ctxs", [[1537], [512, 513, 1024, 1025, 0, 1700], [600] * 20])
def test_one_launch_decode_step_over_chunks(dev, monkeypatch, ctxs):
    """The decode step that forms its own query, key and value: outputs and caches with and without the workspace."""
    torch.manual_seed(len(ctxs))
    print("case decode step", ctxs, flush=True)
    hq, hkv, L, B = 8, 2, 1728, len(ctxs)
    w = (1 + 0.1 * torch.randn(D, device=dev)).to(torch.bfloat16)
    inv = O.rope_inv_freq(D, 1e6).to(dev)
    qkv = torch.randn((B, (hq + 2 * hkv) * D), device=dev).to(torch.bfloat16)
    kc = torch.randn((B, hkv, L, D), device=dev).to(torch.bfloat16)
    vt = torch.randn((B, hkv, D, L), device=dev).to(torch.bfloat16)
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=dev)
    assert _lib.lib().bi_attention_workspace_bytes(B, 1, hq, hkv, L) > 0
    k1, v1, k2, v2 = kc.clone(), vt.clone(), kc.clone(), vt.clone()
    live = ctx > 0
    a = ops.bi_attention_decode_qkv(qkv, w, w, inv, k1, v1, ctx, hq, hkv, SCALE, 1e-6)
    _no_workspace(monkeypatch)
    b = ops.bi_attention_decode_qkv(qkv, w, w, inv, k2, v2, ctx, hq, hkv, SCALE, 1e-6)
    assert torch.equal(a[live], b[live]) and torch.equal(k1, k2) and torch.equal(v1, v2)


def _guarded(nbytes, dev):
    """Scratch of nbytes with a pattern behind it that no kernel may touch."""
    return torch.full((nbytes + 4096,), 0xA5, dtype=torch.uint8, device=dev)


def _untouched(ws, nbytes):
    return bool((ws[nbytes:] == 0xA5).all())


@pytest.mark.parametrize("over", [1, 31, 513, 5000])
@pytest.mark.parametrize("which", [1, 3])
def test_a_sequence_past_its_cache_spoils_no_other(dev, which, over):
    """ctx_len is device data and may run off the cache (a finished sequence in a replayed graph): the chunk states of the
    other rows and the memory behind the workspace stay what they are.  `which`: in the middle of the batch, and the last."""
    print("case past the cache", which, over, flush=True)
    hq, hkv, L, B = 8, 2, 2048, 4
    gen = torch.Generator(device=dev).manual_seed(over)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    qkv, kc, vt = rnd(B, (hq + 2 * hkv) * D), rnd(B, hkv, L, D), rnd(B, hkv, D, L)
    w, inv = (1 + 0.1 * torch.randn(D, generator=gen, device=dev)).to(torch.bfloat16), O.rope_inv_freq(D, 1e6).to(dev)
    lib, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    nbytes = lib.bi_attention_workspace_bytes(B, 1, hq, hkv, L)
    others = [b for b in range(B) if b != which]
    one, starts = torch.ones(B, dtype=torch.int32, device=dev), torch.arange(B, dtype=torch.int32, device=dev)
    q = qkv[:, : hq * D].contiguous()
    got = []
    for last in (L, L + over):
        ctxs = [700, 2048, 1500, 600]
        ctxs[which] = last
        ctx = torch.tensor(ctxs, dtype=torch.int32, device=dev)
        k1, v1, ws = kc.clone(), vt.clone(), _guarded(nbytes, dev)
        fused, plain = torch.zeros((B, hq, D), dtype=torch.bfloat16, device=dev), torch.zeros((B, hq, D), dtype=torch.bfloat16, device=dev)
        assert lib.bi_attention_decode_qkv_ws_bf16(qkv.data_ptr(), qkv.stride(0), w.data_ptr(), w.data_ptr(), inv.data_ptr(), k1.data_ptr(),
                                                   v1.data_ptr(), fused.data_ptr(), ctx.data_ptr(), B, hq, hkv, D, L, SCALE, 1e-6,
                                                   ws.data_ptr(), nbytes, s) == _lib.TBIK_OK
        assert _untouched(ws, nbytes)
        assert lib.bi_attention_ws_bf16(q.data_ptr(), kc.data_ptr(), vt.data_ptr(), plain.data_ptr(), starts.data_ptr(), one.data_ptr(),
                                        ctx.data_ptr(), B, 1, hq, hkv, D, L, SCALE, ws.data_ptr(), nbytes, s) == _lib.TBIK_OK
        assert _untouched(ws, nbytes)
        got.append((fused[others], plain[others], k1[others], v1[others]))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("hq,hkv,qlens,max_q_len", [
    (8, 2, [1, 4, 1, 3], 1),          # decode tiles: room for 16 / 4 queries
    (4, 4, [2, 16, 1, 9], 2),         # ... for 16
    (8, 2, [20, 32, 17, 30], 20),     # two blocks of 16
])
def test_more_queries_than_the_call_says(dev, hq, hkv, qlens, max_q_len):
    """q_len is device data: rows beyond the caller's max_q_len that still fit the tiles come out as without the workspace,
    and nothing is written outside it."""
    print("case more queries", hq, hkv, qlens, max_q_len, flush=True)
    gen = torch.Generator(device=dev).manual_seed(max_q_len)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    L, B = 2048, len(qlens)
    q, kc, vt = rnd(sum(qlens), hq, D), rnd(B, hkv, L, D), rnd(B, hkv, D, L)
    starts, n, ctx = i32([sum(qlens[:i]) for i in range(B)]), i32(qlens), i32([2048, 1700, 600, 1025])
    lib, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    nbytes = lib.bi_attention_workspace_bytes(B, max_q_len, hq, hkv, L)
    assert nbytes > 0
    ws, out, want = _guarded(nbytes, dev), torch.zeros_like(q), torch.zeros_like(q)
    for o, w, wb in ((want, None, 0), (out, ws.data_ptr(), nbytes)):
        assert lib.bi_attention_ws_bf16(q.data_ptr(), kc.data_ptr(), vt.data_ptr(), o.data_ptr(), starts.data_ptr(), n.data_ptr(),
                                        ctx.data_ptr(), B, max_q_len, hq, hkv, D, L, SCALE, w, wb, s) == _lib.TBIK_OK
    assert _untouched(ws, nbytes) and torch.equal(out, want)


@pytest.mark.parametrize("ctx", [40, 520, 1100])
def test_scores_at_the_ends_of_fp32(dev, monkeypatch, ctx):
    """Rows whose scores all lie near the lowest finite fp32 (the mean of the values, exactly 1), rows with some keys at
    -inf (without weight, a whole chunk of them too), and a row with a NaN: every kernel, with and without the workspace."""
    print("case extreme scores", ctx, flush=True)
    hq, hkv, L = 8, 2, 2048
    q = torch.zeros((1, hq, D), dtype=torch.bfloat16, device=dev)
    q[:, :, 0] = 1
    one, start, n = (torch.tensor([v], dtype=torch.int32, device=dev) for v in (1, 0, ctx))
    scale = 1.3862943649291992                              # times log2(e) in fp32: exactly 2, so that large scores scale exactly
    low = torch.tensor(-1.6e38).to(torch.bfloat16).item()   # -3.2e38 after it
    cases = {"low": low, "some": 0.0, "nan": 0.0}
    for name, fill in cases.items():
        k = torch.zeros((L, D))
        k[:, 0] = fill
        v = torch.ones((L, D))
        if name == "some":
            k[: min(ctx - 8, 1024), 0] = -math.inf          # the whole of the first chunks, or all but a few keys
            v[: min(ctx - 8, 1024)] = 7.0
        if name == "nan":
            k[ctx // 2, 0] = math.nan
        for length in (L, L + 4):
            kc = torch.zeros((1, hkv, length, D), dtype=torch.bfloat16, device=dev)
            vt = torch.zeros((1, hkv, D, length), dtype=torch.bfloat16, device=dev)
            kc[0, :, :L], vt[0, :, :, :L] = k.to(torch.bfloat16).to(dev), v.t().to(torch.bfloat16).to(dev)
            for shared in (True, False):
                with monkeypatch.context() as m:
                    if not shared:
                        _no_workspace(m)
                    got = ops.bi_attention_bf16(q, kc, vt, start, one, n, 1, scale)
                    wide = ops.bi_attention_bf16(q.expand(20, hq, D).contiguous(), kc, vt, start, one * 20, n, 20, scale)[-1:]
                for o in (got, wide):
                    assert torch.isnan(o).all() if name == "nan" else torch.equal(o, torch.ones_like(o)), (name, length, shared)
