"""The row-wise operators by the extension's short way and by the long one: the same results, and the same refusals, over the
forms of input that the long way takes."""
import numpy as np
import pytest
import torch

from llm_reproducibility_amd import ops

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


def _forms(dev, dt):
    """name -> matrix: plain ones, rows further apart, rows that no kernel reads in place, other ranks, empty, subclasses."""
    g = torch.Generator(device=dev).manual_seed(3)
    r = lambda *s: torch.randn(s, generator=g, device=dev).to(dt)  # noqa: E731
    yield "plain", r(5, 256)
    yield "one row", r(1, 64)
    yield "row of a wide one", r(3, 512)[1:2, 128:384]
    yield "far rows", r(5, 512)[:, :256]
    yield "odd stride", r(5, 260)[:, :256]
    yield "misaligned", r(5 * 256 + 1)[1:].view(5, 256)
    yield "transposed", r(256, 32).t()
    yield "expanded", r(1, 256).expand(4, 256)
    yield "every second column", r(5, 512)[:, ::2]
    yield "columns no multiple of eight", r(5, 252)
    yield "three dimensions", r(2, 3, 256)
    yield "a vector", r(256)
    yield "no rows", r(0, 256)
    yield "parameter", torch.nn.Parameter(r(5, 256))
    yield "subclass", r(5, 256).as_subclass(Sub)
    yield "on the CPU", r(5, 256).cpu()


def _outcome(f):
    try:
        got = f()
    except Exception as e:  # noqa: BLE001
        return type(e)
    return [(t.shape, t.dtype, t.stride(), t.requires_grad, t.detach().as_subclass(torch.Tensor).clone()) for t in (got if isinstance(got, (list, tuple)) else [got])]


def _same(a, b):
    if isinstance(a, type) or isinstance(b, type):
        return a is b
    return len(a) == len(b) and all(x[:4] == y[:4] and torch.equal(x[4], y[4]) for x, y in zip(a, b))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32, torch.int32])
def test_short_way_and_long_way(dev, dt):
    for name, x in _forms(dev, dt if dt.is_floating_point else torch.float32):
        if not dt.is_floating_point:
            x = x.detach().to(dt)
        n = x.shape[-1]
        weights = {"none": None, "plain": torch.ones(n, device=dev, dtype=x.dtype) * 2, "other type": torch.ones(n, device=dev, dtype=torch.float64),
                   "every second": torch.arange(2 * n, device=dev).to(x.dtype)[::2], "parameter": torch.nn.Parameter(torch.ones(n, device=dev, dtype=torch.bfloat16))}
        for wn, w in weights.items():
            print("case", dt, name, wn, flush=True)
            assert _same(_outcome(lambda: ops.bi_rmsnorm(x, w, 1e-5)), _outcome(lambda: ops._bi_rmsnorm_impl(x, w, 1e-5)))
            for res in (x.detach().clone(), x.detach()[..., : n]):
                assert _same(_outcome(lambda: ops.bi_add_rmsnorm(x, res, w, 1e-5)), _outcome(lambda: ops._bi_add_rmsnorm_impl(x, res, w, 1e-5)))
        assert _same(_outcome(lambda: ops.bi_silu_mul(x)), _outcome(lambda: ops._bi_silu_mul_impl(x)))
        for dim in (-1, 0, x.ndim - 1):
            for keep in (False, True):
                assert _same(_outcome(lambda: ops.bi_mean_dim(x, dim, keep)), _outcome(lambda: ops._bi_mean_dim_impl(x, dim, keep)))
        for soft in (False, True):
            for f32 in (False, True):
                assert _same(_outcome(lambda: ops.bi_log_softmax(x, soft, f32)), _outcome(lambda: ops._bi_log_softmax_impl(x, soft, f32)))


def test_plain_calls_take_the_short_way(dev):
    x = torch.randn((7, 4096), device=dev, dtype=torch.bfloat16)
    f, w = ops._fast(), torch.ones(4096, device=dev, dtype=torch.bfloat16)
    got = [f.rms_norm(x, w, 1e-6), f.add_rms_norm(x, x, None, 1e-6), f.silu_mul(x), f.mean_last(x, True), f.log_softmax(x, False, True)]
    assert all(g is not None for g in got)
    assert f.rms_norm(x, w, 1) is None and f.rms_norm(x.float(), w, 1e-6) is None and f.mean_last(x.t(), False) is None
    with pytest.raises(Exception):
        torch.vmap(lambda v: ops.bi_rmsnorm(v, w, 1e-6))(torch.stack([x, x]))   # as the long way: no batching rule


def test_on_another_stream_and_in_a_graph(dev):
    x, w = torch.randn((9, 2048), device=dev, dtype=torch.bfloat16), torch.ones(2048, device=dev, dtype=torch.bfloat16)
    want = ops._bi_rmsnorm_impl(x, w, 1e-6)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = ops.bi_rmsnorm(x, w, 1e-6)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.equal(got, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = ops.bi_rmsnorm(x, w, 1e-6)
    for k in range(3):
        x.normal_()
        g.replay()
        assert torch.equal(out, ops._bi_rmsnorm_impl(x, w, 1e-6)), k


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_flags_that_are_no_bool(dev, dt):
    """0, 1, None and numpy's bools count as what they are true for, as on the long way."""
    x = torch.randn((5, 256), generator=torch.Generator(device=dev).manual_seed(4), device=dev).to(dt)
    for one in (0, 1, 2, np.bool_(False), np.bool_(True), None):
        truth = bool(one)
        assert _same(_outcome(lambda: ops.bi_mean_dim(x, -1, one)), _outcome(lambda: ops.bi_mean_dim(x, -1, truth)))
        assert _same(_outcome(lambda: ops.bi_log_softmax(x, False, one)), _outcome(lambda: ops.bi_log_softmax(x, False, truth)))
        want = _outcome(lambda: ops._bi_log_softmax_impl(x, one, False))    # (None is a TypeError there)
        assert _same(_outcome(lambda: ops.bi_log_softmax(x, one)), want)
        if one is not None:
            assert _same(want, _outcome(lambda: ops.bi_log_softmax(x, truth)))
