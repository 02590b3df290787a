"""The workloads this library is measured on: what its users have it do, over the range of sizes they do it at.

Five kinds of work, each through the public entry points:

  reduce   the row-wise operators between the matmuls: `rms_norm` (with and without residual), `bi_silu_mul`, `mean`
  row      a row-split layer (o_proj, down_proj): the tree-ordered matmul, as a whole or as simulated tensor-parallel
           shards with the shard tree, `nn.Linear` weights or a row-major right operand
  linear   a column-split or replicated layer through torch's own operators in batch-invariant mode, forward only
           (serving, scoring) or forward and backward (training on the kernels that serve)
  logprob  log-probabilities of every token of the vocabulary through `torch.log_softmax` in batch-invariant mode
  layers   consecutive decoder layers of an engine that holds the KV caches: decode, prefill and chunked prefill

Sizes are those of the models named in this repository's benchmark and tests (Qwen3-8B: hidden 4096, 32/8 heads,
intermediate 12288, vocabulary 151936; Qwen3-32B's row-split layers: 8192 -> 5120 and 25600 -> 5120; the 1.7B-sized
self-check 6144 -> 2048).  Weights are N(0, 0.02), activations N(0, 1) or SiLU-gated, keys unit-normal as they are
behind the per-head norm.
"""
import math

import torch

from llm_reproducibility_amd import ops
from llm_reproducibility_amd.bio import batch_invariant_ops as bio
from llm_reproducibility_amd.layers import SimulatedTPRowLinear
from llm_reproducibility_amd.patch.patch_training_inference_align import compute_inv_freq
from llm_reproducibility_amd.tbik import choose_leaf_k, matmul_tp_persistent, tree_combine

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
HIDDEN, Q_HEADS, KV_HEADS, HEAD_DIM, INTER, VOCAB = 4096, 32, 8, 128, 12288, 151936
QKV = (Q_HEADS + 2 * KV_HEADS) * HEAD_DIM
EPS = 1e-6
# K, N of the row-split layers (o_proj and down_proj of the 8B and 32B models, down_proj of the self-check)
ROW_SHAPES = ((4096, 4096), (12288, 4096), (8192, 5120), (25600, 5120), (6144, 2048))
# K, N of the other layers: qkv, merged gate/up, square, lm_head
LINEAR_SHAPES = ((4096, QKV), (4096, 2 * INTER), (4096, 4096), (4096, VOCAB))


def listed():
    return [
        # the smallest call of a decode step: add-RMSNorm of a handful of rows, all launch and host time
        dict(name="norm 7 rows", kind="reduce", op="add_rms_norm", rows=7, cols=HIDDEN, dtype="bf16"),
        # one sequence decoding: down_proj of the 8B model streams its weights for one row
        dict(name="row-split 1 row", kind="row", M=1, K=12288, N=4096, dtype="bf16", tp=1, layout="linear"),
        # a mid-sized decode batch on the largest row-split layer there is (leaves of 128, an odd row count)
        dict(name="row-split 32B 49 rows", kind="row", M=49, K=25600, N=5120, dtype="bf16", tp=1, layout="linear"),
        # a prefill batch of 2048 tokens, the headline shape of the benchmark
        dict(name="row-split 2048 rows", kind="row", M=2048, K=12288, N=4096, dtype="bf16", tp=1, layout="linear"),
        # the self-check of a tensor-parallel set-up: K cut into four shards, a plain row-major right operand, fp16
        dict(name="row-split self-check fp16", kind="row", M=1024, K=6144, N=2048, dtype="fp16", tp=4, layout="row_major"),
        # weights kept in 16 bits and computed in fp32, the reproducibility study's third precision, on a small batch
        dict(name="linear fp32", kind="linear", M=256, K=4096, N=4096, dtype="fp32", backward=False),
        # one layer of policy training on the serving kernels: qkv projection, forward and both gradients
        dict(name="linear training", kind="linear", M=2048, K=4096, N=QKV, dtype="bf16", backward=True),
        # scoring a rollout: log-probabilities of a thousand tokens from the logits the model hands over
        dict(name="logprob 1000 tokens", kind="logprob", rows=1000, cols=VOCAB, dtype="bf16"),
        # one chat turn: a single sequence, a short context
        dict(name="decode 1 seq", kind="layers", batch=1, new=1, ctx=577, layers=4),
        # a serving batch with contexts of a few hundred to a thousand tokens
        dict(name="decode 32 seqs", kind="layers", batch=32, new=1, ctx=900, layers=4),
        # long inputs (the latency recipe's 8192 tokens) with few sequences: attention over the cache takes over
        dict(name="decode 8 seqs long", kind="layers", batch=8, new=1, ctx=8200, layers=4),
        # prompts coming in: ragged, up to 4096 tokens, no cached prefix
        dict(name="prefill 3 prompts", kind="layers", batch=3, new=4096, ctx=4096, layers=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cost(case):
    """Memory traffic in bytes that the case is worth, with the matrix rate of its type priced in."""
    w = work(case)
    return max(w["bytes"], w["flops"] / 50 * (16 if case.get("dtype") == "fp32" else 1))


def _draw_once(rng):
    kind = rng.choice(("reduce", "row", "row", "linear", "linear", "logprob", "layers", "layers", "layers"))
    if kind == "reduce":
        op = rng.choice(("rms_norm", "add_rms_norm", "silu_mul", "mean"))
        dtype = rng.choice(("bf16", "fp16", "fp32")) if op == "mean" else rng.choice(("bf16", "bf16", "fp16"))
        return dict(kind=kind, op=op, rows=_log_int(rng, 1, 8192), cols=INTER if op == "silu_mul" else rng.choice((2048, 4096, 5120)), dtype=dtype)
    if kind == "row":
        K, N = rng.choice(ROW_SHAPES)
        return dict(kind=kind, M=_log_int(rng, 1, 4096), K=K, N=N, dtype=rng.choice(("bf16",) * 4 + ("fp16", "fp32")),
                    tp=rng.choice((1, 1, 2, 4, 8)), layout=rng.choice(("linear",) * 3 + ("row_major",)))
    if kind == "linear":
        K, N = rng.choice(LINEAR_SHAPES)
        backward = N != VOCAB and rng.random() < 0.4
        return dict(kind=kind, M=_log_int(rng, 64 if backward else 1, 128 if N == VOCAB else 4096), K=K, N=N,
                    dtype=rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32")), backward=backward)
    if kind == "logprob":
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), cols=rng.choice((VOCAB, VOCAB, 32000, 50257)), dtype=rng.choice(("bf16", "fp32")))
    mode = rng.choice(("decode", "decode", "prefill", "chunk"))
    if mode == "decode":
        batch = _log_int(rng, 1, 128)
        return dict(kind=kind, batch=batch, new=1, ctx=_log_int(rng, 64, 16384), layers=4)
    new = _log_int(rng, 16, 4096)
    ctx = new if mode == "prefill" else new + _log_int(rng, 64, 8192)
    return dict(kind=kind, batch=_log_int(rng, 1, 16), new=new, ctx=ctx, layers=2)


def draw(rng):
    largest = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        # at most 2^21 cached positions in all layers (8 GiB), so that a state leaves room for others
        if _cost(case) <= largest and case.get("batch", 0) * case.get("ctx", 0) * case.get("layers", 0) <= 1 << 21:
            return case


# ------------------------------------------------------------------------------------------------------------------
def _lengths(case):
    """(new tokens, context) of every sequence: ragged between two thirds of the stated length and all of it, which the
    first sequence has."""
    got = []
    for b in range(case["batch"]):
        cut = (b * 5 % 8) / 8 * 0.375 if case["batch"] > 1 else 0.0
        new = max(1, int(case["new"] * (1 - cut)))
        ctx = new if case["new"] == case["ctx"] else max(new, int(case["ctx"] * (1 - cut)))
        got.append((new, ctx))
    return got


def _layer_weights():
    return QKV * HIDDEN + 2 * INTER * HIDDEN + HIDDEN * Q_HEADS * HEAD_DIM + HIDDEN * INTER


def work(case):
    kind = case["kind"]
    if kind == "layers":
        lens = _lengths(case)
        tokens = sum(n for n, _ in lens)
        keys = sum(c for _, c in lens)
        pairs = sum(n * (c - n) + n * (n + 1) // 2 for n, c in lens)
        per_layer_bytes = 2 * _layer_weights() + 4 * keys * KV_HEADS * HEAD_DIM
        per_layer_flops = 2 * tokens * _layer_weights() + 4 * pairs * Q_HEADS * HEAD_DIM
        return {"bytes": case["layers"] * per_layer_bytes + 6 * tokens * HIDDEN, "flops": case["layers"] * per_layer_flops}
    size = DTYPES[case["dtype"]].itemsize
    if kind == "reduce":
        n = case["rows"] * case["cols"]
        if case["op"] == "mean":
            return {"bytes": size * (n + case["rows"]), "flops": n}
        if case["op"] == "silu_mul":
            return {"bytes": size * 3 * n, "flops": 5 * n}
        return {"bytes": size * ((4 if case["op"] == "add_rms_norm" else 2) * n + case["cols"]), "flops": 5 * n}
    if kind == "logprob":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * size * n, "flops": 4 * n}
    M, K, N = case["M"], case["K"], case["N"]
    if kind == "row":
        return {"bytes": size * (M * K + K * N + M * N), "flops": 2 * M * K * N}
    if case["backward"]:
        # in: activations, weights, gradient of the output; out: product, both gradients
        return {"bytes": size * 2 * (M * K + K * N + M * N), "flops": 6 * M * K * N}
    return {"bytes": size * (M * K + K * N + M * N), "flops": 2 * M * K * N}


def tolerance(case):
    """Relative errors between correct implementations at the stated precision.  Measured against 64-bit arithmetic on
    the same inputs: 1.7e-3 (mm) to 7e-3 (a tree of 200 bf16 leaves) in bf16, an eighth of that in fp16, 3e-6 for sums
    of fp32 products.  Four layers compound their roundings to 1.4e-2 on each side of a comparison.  `differ` does not
    apply: no case returns whole numbers."""
    if case["kind"] == "layers":
        return {"rel": 3e-2}
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}


# ------------------------------------------------------------------------------------------------------------------
def _normal(gen, shape, dtype, scale=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype).mul_(scale)


def _prepare_layers(case, gen):
    bf16 = torch.bfloat16
    lens = _lengths(case)
    tokens = sum(n for n, _ in lens)
    max_len = (max(c for _, c in lens) + 31) // 32 * 32
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(
            input_norm=_normal(gen, HIDDEN, bf16, 0.1).add_(1), post_norm=_normal(gen, HIDDEN, bf16, 0.1).add_(1),
            q_norm=_normal(gen, HEAD_DIM, bf16, 0.1).add_(1), k_norm=_normal(gen, HEAD_DIM, bf16, 0.1).add_(1),
            qkv=_normal(gen, (QKV, HIDDEN), bf16, 0.02), gate_up=_normal(gen, (2 * INTER, HIDDEN), bf16, 0.02),
            o_proj=SimulatedTPRowLinear(_normal(gen, (HIDDEN, Q_HEADS * HEAD_DIM), bf16, 0.02), 1),
            down_proj=SimulatedTPRowLinear(_normal(gen, (HIDDEN, INTER), bf16, 0.02), 1),
            k_cache=_normal(gen, (case["batch"], KV_HEADS, max_len, HEAD_DIM), bf16),
            vt_cache=_normal(gen, (case["batch"], KV_HEADS, HEAD_DIM, max_len), bf16)))
    starts = [0]
    for n, _ in lens[:-1]:
        starts.append(starts[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    positions = torch.cat([torch.arange(c - n, c) for n, c in lens]).cuda()
    seq = torch.cat([torch.full((n,), b) for b, (n, _) in enumerate(lens)]).cuda()
    return dict(layers=layers, final_norm=_normal(gen, HIDDEN, bf16, 0.1).add_(1), x=_normal(gen, (tokens, HIDDEN), bf16),
                q_start=i32(starts), q_len=i32([n for n, _ in lens]), ctx_len=i32([c for _, c in lens]),
                max_new=max(n for n, _ in lens), positions=positions, seq=seq,
                inv_freq=compute_inv_freq(HEAD_DIM, 1e6, torch.device("cuda")))


def prepare(case, seed):
    bio.enable_batch_invariant_mode()       # once per process, as a serving or training program does at its start
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "layers":
        return dict(case=case, **_prepare_layers(case, gen))
    dt = DTYPES[case["dtype"]]
    if kind == "reduce":
        cols = case["cols"] * (2 if case["op"] == "silu_mul" else 1)
        return dict(case=case, x=_normal(gen, (case["rows"], cols), dt), residual=_normal(gen, (case["rows"], cols), dt, 4.0),
                    weight=_normal(gen, cols, dt, 0.1).add_(1))
    if kind == "logprob":
        return dict(case=case, logits=_normal(gen, (case["rows"], case["cols"]), dt, 1.3))
    M, K, N = case["M"], case["K"], case["N"]
    weight = _normal(gen, (N, K), dt, 0.02)
    x = _normal(gen, (M, K), dt)
    if kind == "row":
        x = torch.nn.functional.silu(x) * _normal(gen, (M, K), dt)
        if case["layout"] == "row_major":
            return dict(case=case, x=x, leaf=choose_leaf_k(K), B=weight.t().contiguous())
        return dict(case=case, x=x, layer=SimulatedTPRowLinear(weight, case["tp"]))
    if case["backward"]:
        return dict(case=case, x=x.requires_grad_(), weight=weight.requires_grad_(), grad=_normal(gen, (M, N), dt, 0.01))
    return dict(case=case, x=x, weight=weight)


def _run_layers(s):
    """The layers as an engine composes them: norms and activations ride inside the projections next to them."""
    x, residual, h = s["x"], None, None
    scale = 1.0 / math.sqrt(HEAD_DIM)
    layers = s["layers"]
    for i, w in enumerate(layers):
        few = x.shape[0] <= 4
        if few:
            qkv, new = ops.rmsnorm_gemm(x, w["input_norm"], EPS, residual, w["qkv"].t())
            residual = x if residual is None else new
        else:
            if h is None:
                h, residual = bio.rms_norm(x, w["input_norm"], EPS), x
            qkv = bio.matmul_persistent(h, w["qkv"].t())
        if s["max_new"] == 1:
            a = ops.bi_attention_decode_qkv(qkv, w["q_norm"], w["k_norm"], s["inv_freq"], w["k_cache"], w["vt_cache"], s["ctx_len"],
                                            Q_HEADS, KV_HEADS, scale, EPS)
        else:
            q = ops.bi_qk_norm_rope_cache_bf16(qkv, w["q_norm"], w["k_norm"], s["inv_freq"], s["positions"], s["seq"], w["k_cache"],
                                               w["vt_cache"], Q_HEADS, KV_HEADS, EPS)
            a = ops.bi_attention_bf16(q, w["k_cache"], w["vt_cache"], s["q_start"], s["q_len"], s["ctx_len"], s["max_new"], scale)
        a = a.reshape(-1, Q_HEADS * HEAD_DIM)
        if few:
            x = w["o_proj"](a)
            gate_up, residual = ops.rmsnorm_gemm(x, w["post_norm"], EPS, residual, w["gate_up"].t())
            x = w["down_proj"].forward_gated(gate_up)
        else:
            h, residual = w["o_proj"].forward_add_norm(a, residual, w["post_norm"], EPS)
            act = ops.gemm_silu_mul(h, w["gate_up"])
            following = layers[i + 1]["input_norm"] if i + 1 < len(layers) else s["final_norm"]
            h, residual = w["down_proj"].forward_add_norm(act, residual, following, EPS)
    if h is None:
        h, residual = bio.rms_norm(x, s["final_norm"], EPS, residual)
    return {"hidden": h, "residual": residual, "keys": [w["k_cache"] for w in layers], "values": [w["vt_cache"] for w in layers]}


@torch.no_grad()
def _run_row(s):
    if "layer" in s:
        return s["layer"](s["x"])
    # each simulated rank's product from its slices of K, then the shard tree
    x, B, tp = s["x"], s["B"], s["case"]["tp"]
    ks = x.shape[1] // tp
    parts = [matmul_tp_persistent(x[:, r * ks:(r + 1) * ks], B[r * ks:(r + 1) * ks], leaf_k=s["leaf"]) for r in range(tp)]
    return parts[0] if tp == 1 else tree_combine(parts)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "layers":
        return _run_layers(state)
    if kind == "row":
        return _run_row(state)
    if kind == "logprob":
        return torch.log_softmax(state["logits"], dim=-1)
    if kind == "linear":
        if case["backward"]:
            out = torch.nn.functional.linear(state["x"], state["weight"])
            gx, gw = torch.autograd.grad(out, (state["x"], state["weight"]), state["grad"])
            return {"out": out.detach(), "grad_x": gx, "grad_weight": gw}
        return torch.nn.functional.linear(state["x"], state["weight"])
    op = case["op"]
    if op == "rms_norm":
        return bio.rms_norm(state["x"], state["weight"], EPS)
    if op == "add_rms_norm":
        out, residual = bio.rms_norm(state["x"], state["weight"], EPS, state["residual"])
        return {"out": out, "residual": residual}
    if op == "silu_mul":
        return ops.bi_silu_mul(state["x"])
    return torch.mean(state["x"], dim=-1)
