"""The forms of the grouped attention kernel (one or two blocks of queries per wavefront, loaders beside them or not, two or
four slots of 64 keys, a chunk per work-group) at caches that end in the middle of a slot: the bits of the one-wave kernel, and the float64 oracle's values."""
import ctypes
import math

import pytest
import torch

from llm_reproducibility_amd import _lib, ops
from oracle import tbik_oracle as O

pytestmark = pytest.mark.gpu
D, SCALE = 128, 1.0 / math.sqrt(128)


def _at_end_of_nan(t):
    """The tensor in memory that goes on with NaNs.  They show a value that is taken from behind the whole cache, where its last
    channel row goes on, even with the weight 0; a key from there is masked before it can show, and behind every other row lies the
    next one (a NaN there would be a visible key's)."""
    buf = torch.full((t.numel() + 4096,), math.nan, dtype=t.dtype, device=t.device)
    buf[: t.numel()] = t.reshape(-1)
    return buf[: t.numel()].view(t.shape)


# query heads, KV heads, sequences, longest number of new tokens, cache length; then the form: work-groups per row, slots, queries per
# work-group, blocks of 16 per wavefront, wavefronts that load
@pytest.mark.parametrize("hq,hkv,B,new,L,form", [
    (32, 8, 171, 33, 96, (1, 2, 32, 2, 0)), (32, 8, 28, 33, 1120, (1, 2, 32, 2, 0)), (16, 8, 260, 33, 96, (1, 2, 64, 2, 0)),
    (16, 8, 41, 33, 1120, (1, 2, 64, 2, 0)), (8, 8, 260, 70, 96, (1, 2, 128, 2, 0)), (8, 8, 41, 70, 1120, (1, 2, 128, 2, 0)),
    (32, 4, 60, 300, 544, (1, 2, 32, 2, 0)), (64, 8, 2, 1500, 1568, (1, 2, 32, 2, 0)),                 # two blocks of queries per wavefront
    (64, 8, 20, 33, 96, (1, 2, 16, 1, 0)), (32, 8, 36, 17, 1120, (1, 2, 16, 1, 0)), (16, 8, 4, 600, 1120, (1, 2, 32, 1, 0)),
    (8, 8, 8, 300, 544, (1, 2, 64, 1, 0)),                                                             # one
    (64, 8, 20, 33, 1120, (1, 2, 16, 1, 4)), (64, 8, 5, 50, 1120, (1, 2, 16, 1, 4)), (64, 8, 8, 25, 96, (1, 2, 16, 1, 4)),
    (32, 8, 28, 33, 96, (1, 2, 16, 1, 4)), (32, 8, 1, 1000, 1120, (1, 2, 16, 1, 4)), (16, 8, 2, 40, 160, (1, 2, 16, 1, 4)),
    (16, 8, 12, 33, 160, (1, 2, 32, 1, 4)), (16, 8, 1, 1000, 1120, (1, 2, 32, 1, 4)), (16, 4, 35, 37, 96, (1, 2, 16, 1, 4)), (4, 4, 2, 20, 32, (1, 2, 16, 1, 4)),
    (4, 4, 33, 50, 96, (1, 2, 64, 1, 4)), (4, 4, 1, 1000, 1120, (1, 2, 64, 1, 4)),                     # one, loaders
    (32, 8, 3, 100, 1120, (1, 4, 16, 1, 4)), (32, 8, 5, 50, 1120, (1, 4, 16, 1, 4)), (16, 8, 10, 50, 1120, (1, 4, 32, 1, 4)),
    (4, 4, 33, 64, 1120, (1, 4, 64, 1, 4)), (64, 8, 9, 33, 2080, (1, 4, 16, 1, 4)),                    # one, four slots
    (32, 8, 1, 40, 1120, (3, 2, 16, 1, 4)), (3, 3, 2, 20, 1568, (4, 2, 64, 1, 4)), (16, 8, 1, 40, 1120, (3, 2, 32, 1, 4)),
    (64, 8, 1, 17, 1120, (3, 2, 16, 1, 0)),                                                            # a chunk per work-group
])
def test_forms_at_odd_cache_lengths(dev, hq, hkv, B, new, L, form):
    print("case group forms", hq, hkv, B, new, L, flush=True)
    gen = torch.Generator(device=dev).manual_seed(hq + B + L)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    new = min(new, L)
    lib, info = _lib.lib(), (ctypes.c_int * 6)()
    assert lib.bi_attention_plan_info(B, new, hq, hkv, L, lib.bi_attention_workspace_bytes(B, new, hq, hkv, L), info) == _lib.TBIK_OK
    assert tuple(info) == (1, *form)
    qlens = [(new, 1, min(17, new), min(33, new), max(new - 1, 1))[b % 5] for b in range(B)]
    ctxs = [max(n, (L, L - 31, L - 32, L // 2 + 1, 64, L - 63)[b % 6]) for b, n in enumerate(qlens)]
    ctxs[-1] = L
    starts = [sum(qlens[:i]) for i in range(B)]
    q, kc, vt = rnd(sum(qlens), hq, D), _at_end_of_nan(rnd(B, hkv, L, D)), _at_end_of_nan(rnd(B, hkv, D, L))
    args = (i32(starts), i32(qlens), i32(ctxs), new, SCALE)
    got = ops.bi_attention_bf16(q, kc, vt, *args)
    pad = torch.nn.functional.pad
    assert torch.equal(ops.bi_attention_bf16(q, pad(kc, (0, 0, 0, 4)), pad(vt, (0, 4)), *args), got)   # the one-wave kernel
    for b in {0, B - 1}:
        k, v = kc[b, :, : ctxs[b]].transpose(0, 1).cpu(), vt[b, :, :, : ctxs[b]].permute(2, 0, 1).cpu()
        mine = slice(starts[b], starts[b] + qlens[b])
        assert not O.outside_tolerance(got[mine].cpu(), O.causal_attention(q[mine].cpu(), k, v, SCALE).to(torch.bfloat16)).any()


@pytest.mark.parametrize("hq,hkv", [(2, 2), (4, 2), (8, 2)])
def test_more_rows_than_the_caller_said(dev, monkeypatch, hq, hkv):
    """q_len is device data: rows beyond the workspace's (max_q_len rounded up to 16) stay out of the states of the next sequence."""
    print("case rows beyond", hq, hkv, flush=True)
    gen = torch.Generator(device=dev).manual_seed(hq)
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev).to(torch.bfloat16)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    L, new = 1600, 20
    q, kc, vt = rnd(80, hq, D), rnd(2, hkv, L, D), rnd(2, hkv, D, L)
    args = (i32([0, 60]), i32([60, 20]), i32([1590, 1500]), new, SCALE)
    got = ops.bi_attention_bf16(q, kc, vt, *args)
    monkeypatch.setattr(ops, "_attention_workspace", lambda *a: (None, 0))
    want = ops.bi_attention_bf16(q, kc, vt, *args)
    assert torch.equal(got[:32], want[:32]) and torch.equal(got[60:], want[60:])
