"""Performance cases: the work a rollout-and-loss program has the framework do.

The sizes are Qwen3-0.6B's (hidden 1024, 16 query and 8 KV heads of 128, MLP
3072, vocabulary 151,936, 256-token pages) and those of the repository's own
benchmark and tests; batch, context and token counts are spread over the range
such a program meets.  Every case goes through the public entry points:

  decode_stack   a stack of decoder layers for one new token per sequence,
                 captured once as a HIP graph and replayed, as serving does it
  decode_attn    paged decode attention of one layer, called eagerly
  prefill_attn   varlen attention of a chunk of new tokens over a cached prefix
  prefill_layer  one decoder layer over the new tokens of several prompts
  sample         lm_head + sampling of the next tokens (a top-k, or all entries)
  logprob        lm_head + log-probabilities of given tokens (old / reference
                 policy, the loss step)
  loss           the GRPO loss and its gradient from materialised logits
  train_layer    one decoder layer, forward and backward
  train_step     model forward, GRPO loss, backward: the gradients of all weights
"""
import importlib
import math

import torch

pkg = importlib.import_module("qwen3-naive-inference_amd")

HIDDEN, HEADS, KV_HEADS, HEAD_DIM, INTER, VOCAB, PAGE = 1024, 16, 8, 128, 3072, 151936, 256
EPS, THETA, MAX_POSITION = 1e-6, 1000000.0, 40960
QKV = (HEADS + 2 * KV_HEADS) * HEAD_DIM
LAYER_WEIGHTS = HIDDEN * QKV + HEADS * HEAD_DIM * HIDDEN + 3 * HIDDEN * INTER
SCALE = HEAD_DIM ** -0.5


def listed():
    return [
        # A few interactive requests at short contexts: launches and latency.
        {"name": "decode_stack_4", "kind": "decode_stack", "batch": 4, "lo": 37, "hi": 700, "layers": 8},
        # The 256-sequence rollout in mid-flight: near-equal contexts.
        {"name": "decode_stack_256", "kind": "decode_stack", "batch": 256, "lo": 600, "hi": 680, "layers": 2},
        # 64 ragged long contexts: the attention alone, where the bytes are.
        {"name": "decode_attn_64", "kind": "decode_attn", "batch": 64, "lo": 1024, "hi": 4096},
        # A chunked-prefill step: 16 sequences, 512 new tokens behind a cached prefix of 512.
        {"name": "prefill_attn_16x512", "kind": "prefill_attn", "seqs": 16, "lo": 512, "hi": 512, "prefix": 512},
        # One short prompt: time to first token.
        {"name": "prefill_layer_1x77", "kind": "prefill_layer", "seqs": 1, "lo": 77, "hi": 77, "prefix": 0},
        # A full 2,048-token step of 128-token prompts, as a rollout begins.
        {"name": "prefill_layer_16x128", "kind": "prefill_layer", "seqs": 16, "lo": 128, "hi": 128, "prefix": 0},
        # The generators' default sampling (top 20, T = 0.6) at a serving batch.
        {"name": "sample_64_top20", "kind": "sample", "rows": 64, "top_k": 20, "temperature": 0.6},
        # Rollout sampling: all entries, T = 1, with log-probabilities.
        {"name": "sample_256", "kind": "sample", "rows": 256, "top_k": 0, "temperature": 1.0},
        # Log-probabilities of a micro-batch of finished responses.
        {"name": "logprob_8192", "kind": "logprob", "rows": 8192},
        # The fused loss and the logit gradient for 16 responses of 512 tokens.
        {"name": "loss_16x512", "kind": "loss", "seqs": 16, "tokens": 512},
        # A training micro-batch through one layer, in both directions.
        {"name": "train_layer_8x640", "kind": "train_layer", "seqs": 8, "tokens": 640},
        # A whole training micro-batch: odd length, gradients of every weight.
        {"name": "train_step_2x389", "kind": "train_step", "seqs": 2, "tokens": 389, "layers": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_stack", "decode_attn", "prefill_attn", "prefill_layer", "sample",
                       "logprob", "loss", "train_layer", "train_step"])
    if kind in ("decode_stack", "decode_attn"):
        batch = _log_int(rng, 1, 256)
        hi = _log_int(rng, 40, min(8192, 160000 // batch))
        case = {"kind": kind, "batch": batch, "lo": rng.choice([1, hi // 4 + 1, hi - hi // 10]), "hi": hi}
        if kind == "decode_stack":
            case["layers"] = rng.randint(1, 2)
        return case
    if kind in ("prefill_attn", "prefill_layer"):
        seqs = _log_int(rng, 1, 16)
        hi = _log_int(rng, 5, (8192 if kind == "prefill_attn" else 2048) // seqs)
        prefix = rng.choice([0, 256 * rng.randint(1, 4), rng.randint(1, 1500)])
        return {"kind": kind, "seqs": seqs, "lo": rng.choice([1, hi // 2 + 1, hi]), "hi": hi, "prefix": prefix}
    if kind == "sample":
        return {"kind": kind, "rows": _log_int(rng, 1, 256), "top_k": rng.choice([0, 1, 20, 50]),
                "temperature": rng.choice([0.6, 0.8, 1.0])}
    if kind == "logprob":
        return {"kind": kind, "rows": _log_int(rng, 20, 8192)}
    if kind == "loss":
        return {"kind": kind, "seqs": 4 * rng.randint(1, 4), "tokens": _log_int(rng, 20, 512)}
    seqs = rng.randint(1, 8)
    if kind == "train_layer":
        return {"kind": kind, "seqs": seqs, "tokens": _log_int(rng, 33, min(1152, 5120 // seqs))}
    return {"kind": kind, "seqs": 2 * rng.randint(1, 2), "tokens": _log_int(rng, 33, 360), "layers": rng.randint(1, 2)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(shape, g, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(torch.bfloat16)


def _lengths(case, seed):
    """Per-sequence lengths spread evenly over [lo, hi], in an order of the seed's."""
    n = case.get("batch") or case["seqs"]
    order = torch.randperm(n, generator=torch.Generator().manual_seed(seed)).tolist()
    return [case["hi"] - i * (case["hi"] - case["lo"]) // max(1, n - 1) for i in order]


def _tables(lens, longest, seed):
    """-1 padded page tables over a shuffled pool that would hold len(lens) sequences of `longest` tokens."""
    width = -(-longest // PAGE)
    nb = len(lens) * width
    bt = torch.randperm(nb, generator=torch.Generator().manual_seed(seed)).to(torch.int32).view(-1, width)
    for b, n in enumerate(lens):
        bt[b, -(-n // PAGE):] = -1
    return bt, nb


def _slots(bt, b, first, count):
    t = torch.arange(first, first + count)
    return bt[b].long()[t // PAGE] * PAGE + t % PAGE


def _fill(module, g):
    """Random weights at the scale of a trained model's: norms near one, unit-variance projections."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if "norm" in name:
                p.copy_(torch.rand(p.shape, generator=g, device="cuda") * 0.4 + 0.8)
            else:
                p.copy_(torch.randn(p.shape, generator=g, device="cuda") * (0.25 if "embed" in name else 0.02))


def _module(make, g):
    with torch.device("cuda"):
        m = make().to(torch.bfloat16)
    _fill(m, g)
    return m


def _prepare_decode_stack(case, seed):
    g = _gen(seed)
    layers, batch = case["layers"], case["batch"]
    model = _module(lambda: pkg.Qwen3Model(pkg.Qwen3Config(num_hidden_layers=layers)), g)
    ctx = _lengths(case, seed)
    bt, nb = _tables([c + 1 for c in ctx], case["hi"] + 1, seed)
    k = _randn((layers, nb, PAGE, KV_HEADS, HEAD_DIM), g)
    v = _randn((layers, nb, PAGE, KV_HEADS, HEAD_DIM), g)
    for i, layer in enumerate(model.layers):
        layer.self_attn.k_cache, layer.self_attn.v_cache = k[i], v[i]
    ids = torch.randint(0, VOCAB, (batch,), generator=g, device="cuda")
    slots = torch.cat([_slots(bt, b, c, 1) for b, c in enumerate(ctx)]).to(torch.int32).cuda()
    ctx_dev = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    args = (ids, ctx_dev.long(), ctx_dev, bt.cuda(), slots)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad():
        with torch.cuda.stream(stream):
            model.forward_decode(*args)
        torch.cuda.current_stream().wait_stream(stream)
        with torch.cuda.graph(graph):
            hidden = model.forward_decode(*args)
    return {"kind": case["kind"], "graph": graph, "model": model, "args": args, "ctx": ctx,
            "out": {"hidden": hidden, "k": k, "v": v}}


def _prepare_decode_attn(case, seed):
    g = _gen(seed)
    lens = _lengths(case, seed)
    bt, nb = _tables(lens, case["hi"], seed)
    return {"kind": case["kind"], "q": _randn((case["batch"], HEADS, HEAD_DIM), g), "lens": lens,
            "k": _randn((nb, PAGE, KV_HEADS, HEAD_DIM), g), "v": _randn((nb, PAGE, KV_HEADS, HEAD_DIM), g),
            "seqlens": torch.tensor(lens, dtype=torch.int32, device="cuda"), "tables": bt.cuda()}


def _varlen(case, seed):
    new = _lengths(case, seed)
    prefix = case["prefix"]
    bt, nb = _tables([prefix + n for n in new], prefix + case["hi"], seed)
    zero = torch.zeros(1, dtype=torch.int64)
    cu_q = torch.cat([zero, torch.tensor(new).cumsum(0)]).to(torch.int32).cuda()
    cu_k = torch.cat([zero, (torch.tensor(new) + prefix).cumsum(0)]).to(torch.int32).cuda()
    return new, bt, nb, {"new": new, "prefix": prefix, "tables": bt.cuda(), "cu_q": cu_q, "cu_k": cu_k,
                         "max_q": max(new), "max_k": max(new) + prefix}


def _prepare_prefill_attn(case, seed):
    g = _gen(seed)
    new, _, nb, s = _varlen(case, seed)
    return dict(s, kind=case["kind"], q=_randn((sum(new), HEADS, HEAD_DIM), g),
                k=_randn((nb, PAGE, KV_HEADS, HEAD_DIM), g), v=_randn((nb, PAGE, KV_HEADS, HEAD_DIM), g))


def _prepare_prefill_layer(case, seed):
    g = _gen(seed)
    new, bt, nb, s = _varlen(case, seed)
    layer = _module(lambda: pkg.Qwen3DecoderLayer(pkg.Qwen3Config(num_hidden_layers=1)), g)
    k, v = _randn((nb, PAGE, KV_HEADS, HEAD_DIM), g), _randn((nb, PAGE, KV_HEADS, HEAD_DIM), g)
    layer.self_attn.k_cache, layer.self_attn.v_cache = k, v
    slots = torch.cat([_slots(bt, b, case["prefix"], n) for b, n in enumerate(new)]).to(torch.int32).cuda()
    positions = torch.cat([torch.arange(case["prefix"], case["prefix"] + n) for n in new]).cuda()
    return dict(s, kind=case["kind"], layer=layer, k=k, v=v, slots=slots, positions=positions,
                x=_randn((sum(new), HIDDEN), g, 0.1), residual=_randn((sum(new), HIDDEN), g, 0.25))


def _head(rows, g):
    """Normalised hidden states and an lm_head that gives logits of standard deviation near 3."""
    return _randn((rows, HIDDEN), g), _randn((VOCAB, HIDDEN), g, 0.1)


def _prepare_sample(case, seed):
    g = _gen(seed)
    hidden, weight = _head(case["rows"], g)
    counters = torch.arange(case["rows"], device="cuda") + (torch.randint(0, 1024, (1,), generator=g, device="cuda") << 32)
    return {"kind": case["kind"], "hidden": hidden, "weight": weight, "temperature": case["temperature"],
            "top_k": case["top_k"] or None, "seed": seed, "counters": counters}


def _prepare_logprob(case, seed):
    g = _gen(seed)
    hidden, weight = _head(case["rows"], g)
    return {"kind": case["kind"], "hidden": hidden, "weight": weight,
            "targets": torch.randint(0, VOCAB, (case["rows"],), generator=g, device="cuda")}


def _grpo(seqs, tokens, g, lp, spread):
    """What a rollout leaves beside the tokens: its log-probabilities, the responses' masks, rewards and groups of
    four (of two where there are only two sequences)."""
    lens = torch.randint(max(1, tokens // 8), tokens + 1, (seqs,), generator=g, device="cuda")
    group = 4 if seqs % 4 == 0 else 2
    return {"old": lp + spread * torch.randn(lp.shape, generator=g, device="cuda"),
            "mask": (torch.arange(tokens, device="cuda")[None] < lens[:, None]).float(),
            "rewards": torch.rand(seqs, generator=g, device="cuda"),
            "groups": torch.arange(seqs, device="cuda") // group}


def _prepare_loss(case, seed):
    g = _gen(seed)
    seqs, tokens = case["seqs"], case["tokens"]
    logits = torch.empty((seqs, tokens, VOCAB), dtype=torch.bfloat16, device="cuda")
    ids = torch.empty((seqs, tokens), dtype=torch.int64, device="cuda")
    lp = torch.empty((seqs, tokens), dtype=torch.float32, device="cuda")
    for b in range(seqs):
        logits[b] = _randn((tokens, VOCAB), g, 2.0)
        x = torch.log_softmax(logits[b].float(), -1)
        ids[b] = torch.multinomial(x.exp(), 1, generator=g)[:, 0]
        lp[b] = x.gather(-1, ids[b][:, None])[:, 0]
    return dict(_grpo(seqs, tokens, g, lp, 0.1), kind=case["kind"], logits=logits.requires_grad_(), ids=ids)


def _prepare_train_layer(case, seed):
    g = _gen(seed)
    layer = _module(lambda: pkg.Qwen3DecoderLayer(pkg.Qwen3Config(num_hidden_layers=1)), g)
    shape = (case["seqs"], case["tokens"], HIDDEN)
    return {"kind": case["kind"], "layer": layer, "x": _randn(shape, g, 0.25).requires_grad_(),
            "grad": _randn(shape, g, 0.01)}


def _prepare_train_step(case, seed):
    g = _gen(seed)
    model = _module(lambda: pkg.Qwen3ForCausalLM(pkg.Qwen3Config(
        num_hidden_layers=case["layers"], tie_word_embeddings=False)), g)
    ids = torch.randint(0, VOCAB, (case["seqs"], case["tokens"]), generator=g, device="cuda")
    with torch.no_grad():  # the rollout's log-probabilities: the same weights, rounded elsewhere
        w = {n: p.float() for n, p in model.named_parameters()}
        lp = torch.log_softmax(_model_ref(w, ids, case["layers"])[:, :-1], -1).gather(-1, ids[:, 1:, None])[..., 0]
        lp = torch.cat([torch.zeros_like(lp[:, :1]), lp], 1)
    return dict(_grpo(case["seqs"], case["tokens"], g, lp, 0.02), kind=case["kind"], model=model, ids=ids,
                layers=case["layers"])


_PREPARE = {"decode_stack": _prepare_decode_stack, "decode_attn": _prepare_decode_attn,
            "prefill_attn": _prepare_prefill_attn, "prefill_layer": _prepare_prefill_layer,
            "sample": _prepare_sample, "logprob": _prepare_logprob, "loss": _prepare_loss,
            "train_layer": _prepare_train_layer, "train_step": _prepare_train_step}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_decode_stack(s):
    s["graph"].replay()
    return s["out"]


def _run_decode_attn(s):
    return pkg.kernels.paged_decode_attention(s["q"], s["k"], s["v"], s["seqlens"], s["tables"], SCALE)


def _run_prefill_attn(s):
    return pkg.kernels.varlen_prefill_attention(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], s["max_q"],
                                                s["max_k"], SCALE, True, s["tables"])


def _run_prefill_layer(s):
    with torch.no_grad():
        h, residual = s["layer"].forward_prefill(s["x"], s["positions"], s["cu_q"], s["cu_k"], s["max_q"],
                                                 s["max_k"], s["slots"], s["tables"], s["residual"])
    return {"h": h, "residual": residual, "k": s["k"], "v": s["v"]}


def _run_sample(s):
    tokens, lp = pkg.kernels.lm_head_sample(s["hidden"], s["weight"], s["temperature"], seed=s["seed"],
                                            top_k=s["top_k"], row_counters=s["counters"])
    return {"tokens": tokens, "lp": lp}


def _run_logprob(s):
    lp, lse = pkg.kernels.lm_head_logprob(s["hidden"], s["weight"], s["targets"])
    return {"lp": lp, "lse": lse}


def _run_loss(s):
    s["logits"].grad = None
    loss, lp, adv = pkg.grpo_fused_loss(s["logits"], s["ids"], s["old"], s["mask"], s["rewards"], s["groups"])
    loss.backward()
    return {"loss": loss.detach(), "lp": lp, "adv": adv, "grad": s["logits"].grad}


def _run_train_layer(s):
    s["layer"].zero_grad()
    s["x"].grad = None
    y = s["layer"](s["x"])
    y.backward(s["grad"])
    return {"y": y.detach(), "x": s["x"].grad, "w": {n: p.grad for n, p in s["layer"].named_parameters()}}


def _run_train_step(s):
    model = s["model"]
    model.zero_grad()
    loss, lp, adv = pkg.grpo_fused_loss(model(s["ids"]), s["ids"], s["old"], s["mask"], s["rewards"], s["groups"],
                                        shift=True)
    loss.backward()
    return {"loss": loss.detach(), "lp": lp, "adv": adv, "w": {n: p.grad for n, p in model.named_parameters()}}


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------
def work(case):
    """Weights, K/V rows, inputs and outputs once (bf16); products as multiply + add.  Lengths count with their
    mean."""
    kind = case["kind"]
    row = 2 * HIDDEN
    if kind in ("decode_stack", "decode_attn"):
        n, keys = case["batch"], (case["lo"] + case["hi"]) / 2
        attn = n * keys * 2 * KV_HEADS * HEAD_DIM * 2
        flops = 4.0 * n * keys * HEADS * HEAD_DIM
        if kind == "decode_attn":
            return {"bytes": attn + 4 * n * HEADS * HEAD_DIM, "flops": flops}
        per_layer = attn + 2 * LAYER_WEIGHTS + n * 4 * KV_HEADS * HEAD_DIM
        return {"bytes": case["layers"] * per_layer + 2 * n * row,
                "flops": case["layers"] * (flops + 2.0 * n * LAYER_WEIGHTS)}
    if kind in ("prefill_attn", "prefill_layer"):
        new = (case["lo"] + case["hi"]) / 2
        tokens = case["seqs"] * new
        pairs = case["seqs"] * (new * case["prefix"] + new * (new + 1) / 2)
        flops = 4.0 * pairs * HEADS * HEAD_DIM
        kv = 4 * KV_HEADS * HEAD_DIM
        cached = case["seqs"] * case["prefix"] * kv
        if kind == "prefill_attn":
            return {"bytes": cached + tokens * (kv + 4 * HEADS * HEAD_DIM), "flops": flops}
        return {"bytes": cached + 2 * LAYER_WEIGHTS + tokens * (kv + 4 * row),
                "flops": flops + 2.0 * tokens * LAYER_WEIGHTS}
    if kind in ("sample", "logprob"):
        return {"bytes": 2 * VOCAB * HIDDEN + case["rows"] * (row + 24), "flops": 2.0 * case["rows"] * VOCAB * HIDDEN}
    tokens = case["seqs"] * case["tokens"]
    if kind == "loss":  # the logits are read twice (softmax sums, gradient), the gradient is written
        return {"bytes": 3 * 2 * tokens * VOCAB, "flops": 8.0 * tokens * VOCAB}
    pairs = case["seqs"] * case["tokens"] * (case["tokens"] + 1) / 2
    flops = 14.0 * pairs * HEADS * HEAD_DIM + 6.0 * tokens * LAYER_WEIGHTS
    nbytes = 6 * LAYER_WEIGHTS + tokens * 4 * row
    if kind == "train_layer":
        return {"bytes": nbytes, "flops": flops}
    return {"bytes": case["layers"] * nbytes + 3 * 2 * VOCAB * HIDDEN + 2 * VOCAB * HIDDEN + 3 * 2 * tokens * VOCAB,
            "flops": case["layers"] * flops + 6.0 * tokens * VOCAB * HIDDEN}


def tolerance(case):
    """About four times what a pass measures against 64 bits: bf16 results (0.0017-0.0023 for one attention or the
    logit gradient), layers with several bf16 roundings in a row (0.006; eight of them 0.012), gradients through
    whole layers (0.012); log-probabilities are fp32 over logits rounded to bf16 (0.0004)."""
    return {"rel": {"decode_attn": 8e-3, "prefill_attn": 8e-3, "loss": 7e-3, "decode_stack": 0.03,
                    "prefill_layer": 0.02, "train_layer": 0.03, "train_step": 0.03, "sample": 1.5e-3,
                    "logprob": 1.5e-3}[case["kind"]],
            "differ": 0.01 if case["kind"] == "sample" else 0.0}


# ---------------------------------------------------------------------------
# The same in 64 bits, with plain torch
# ---------------------------------------------------------------------------
def _cos_sin(positions, dtype):
    """The angles as the model defines them: fp32 frequencies times fp32 positions."""
    inv = 1.0 / (THETA ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float) / HEAD_DIM))
    f = torch.outer(torch.arange(0, MAX_POSITION, dtype=torch.float), inv).to(positions.device)[positions]
    return f.cos().to(dtype), f.sin().to(dtype)


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope(x, cos, sin):
    """x [..., heads, 128] with cos / sin [..., 64]."""
    a, b = x[..., :64], x[..., 64:]
    c, s = cos[..., None, :], sin[..., None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _qkv(w, prefix, x, positions):
    q, k, v = (x @ w[prefix + "self_attn.qkv_proj.weight"].T).split([HEADS * HEAD_DIM] + 2 * [KV_HEADS * HEAD_DIM], -1)
    q, k, v = (t.unflatten(-1, (-1, HEAD_DIM)) for t in (q, k, v))
    cos, sin = _cos_sin(positions, x.dtype)
    return (_rope(_norm(q, w[prefix + "self_attn.q_norm.weight"]), cos, sin),
            _rope(_norm(k, w[prefix + "self_attn.k_norm.weight"]), cos, sin), v)


def _attend(q, k, v):
    """Causal attention of the last q.shape[-3] positions: q [..., Tq, 16, 128], k / v [..., Tk, 8, 128]."""
    q, k, v = (t.transpose(-2, -3) for t in (q, k, v))
    k, v = (t.repeat_interleave(HEADS // KV_HEADS, -3) for t in (k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) * SCALE
    tq, tk = s.shape[-2:]
    hidden = torch.ones(tq, tk, dtype=torch.bool, device=s.device).triu(tk - tq + 1)
    return (torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ v).transpose(-2, -3)


def _mlp(w, prefix, x):
    gate, up = (x @ w[prefix + "mlp.gate_up_proj.weight"].T).chunk(2, -1)
    return (torch.nn.functional.silu(gate) * up) @ w[prefix + "mlp.down_proj.weight"].T


def _layer_ref(w, prefix, x):
    """A training layer: x [B, T, hidden]."""
    q, k, v = _qkv(w, prefix, _norm(x, w[prefix + "input_layernorm.weight"]),
                   torch.arange(x.shape[1], device=x.device))
    x = x + _attend(q, k, v).flatten(-2) @ w[prefix + "self_attn.o_proj.weight"].T
    return x + _mlp(w, prefix, _norm(x, w[prefix + "post_attention_layernorm.weight"]))


def _model_ref(w, ids, layers):
    x = w["model.embed_tokens.weight"][ids]
    for i in range(layers):
        x = _layer_ref(w, "model.layers.%d." % i, x)
    return _norm(x, w["model.norm.weight"]) @ w["lm_head.weight"].T


def _loss_ref(lp, s, old, mask):
    """Group-normalised advantages and the clipped token-mean loss."""
    r, adv = s["rewards"].double(), torch.zeros_like(s["rewards"], dtype=torch.float64)
    for p in s["groups"].unique():
        at = s["groups"] == p
        adv[at] = (r[at] - r[at].mean()) / (r[at].std() + 1e-8)
    ratio = (lp - old.double()).exp()
    a = adv[:, None]
    per = -torch.minimum(ratio * a, ratio.clamp(0.8, 1.2) * a)
    return (per * mask.double()).sum() / (mask.double().sum() + 1e-8), adv


def _double(module, grad):
    return {n: p.detach().double().requires_grad_(grad) for n, p in module.named_parameters()}


def _paged(cache, table, n):
    return cache[table[:-(-n // PAGE)].long()].flatten(0, 1)[:n]


def exact(case, seed):
    if case["kind"] == "sample":
        return None  # a draw: whole numbers, and the log-probabilities of what was drawn
    s = prepare(case, seed)
    return globals()["_exact_" + case["kind"]](s)


def _exact_decode_stack(s):
    ids, positions, _, tables, slots = s["args"]
    with torch.no_grad():
        w = _double(s["model"], False)
        k, v = s["out"]["k"].double(), s["out"]["v"].double()
        x = w["embed_tokens.weight"][ids]
        for i in range(k.shape[0]):
            p = "layers.%d." % i
            q, kn, vn = _qkv(w, p, _norm(x, w[p + "input_layernorm.weight"]), positions)
            k[i].flatten(0, 1)[slots.long()], v[i].flatten(0, 1)[slots.long()] = kn, vn
            o = torch.stack([_attend(q[b:b + 1], _paged(k[i], tables[b], n + 1), _paged(v[i], tables[b], n + 1))[0]
                             for b, n in enumerate(s["ctx"])])
            x = x + o.flatten(-2) @ w[p + "self_attn.o_proj.weight"].T
            x = x + _mlp(w, p, _norm(x, w[p + "post_attention_layernorm.weight"]))
        return {"hidden": _norm(x, w["norm.weight"]), "k": k, "v": v}


def _exact_decode_attn(s):
    return torch.stack([_attend(s["q"][b:b + 1].double(), _paged(s["k"], s["tables"][b], n).double(),
                                _paged(s["v"], s["tables"][b], n).double())[0] for b, n in enumerate(s["lens"])])


def _exact_prefill(s, q, k, v):
    out, at = [], 0
    for b, n in enumerate(s["new"]):
        t = s["tables"][b]
        out.append(_attend(q[at:at + n].double(), _paged(k, t, s["prefix"] + n).double(),
                           _paged(v, t, s["prefix"] + n).double()))
        at += n
    return torch.cat(out)


def _exact_prefill_attn(s):
    return _exact_prefill(s, s["q"], s["k"], s["v"])


def _exact_prefill_layer(s):
    with torch.no_grad():
        w = _double(s["layer"], False)
        residual = s["x"].double() + s["residual"].double()
        q, kn, vn = _qkv(w, "", _norm(residual, w["input_layernorm.weight"]), s["positions"])
        k, v = s["k"].double(), s["v"].double()
        k.flatten(0, 1)[s["slots"].long()], v.flatten(0, 1)[s["slots"].long()] = kn, vn
        residual = residual + _exact_prefill(s, q, k, v).flatten(-2) @ w["self_attn.o_proj.weight"].T
        return {"h": _mlp(w, "", _norm(residual, w["post_attention_layernorm.weight"])), "residual": residual,
                "k": k, "v": v}


def _exact_logprob(s):
    x = s["hidden"].double() @ s["weight"].double().T
    lse = torch.logsumexp(x, -1)
    return {"lp": x.gather(-1, s["targets"][:, None])[:, 0] - lse, "lse": lse}


def _exact_loss(s):
    logits = s["logits"].detach().double()
    lse = torch.logsumexp(logits, -1)
    lp = (logits.gather(-1, s["ids"][..., None])[..., 0] - lse).requires_grad_()
    loss, adv = _loss_ref(lp, s, s["old"], s["mask"])
    loss.backward()
    grad = logits.sub_(lse[..., None]).exp_().mul_(-lp.grad[..., None])
    grad.scatter_add_(-1, s["ids"][..., None], lp.grad[..., None])
    return {"loss": loss.detach(), "lp": lp.detach(), "adv": adv, "grad": grad}


def _exact_train_layer(s):
    w, x = _double(s["layer"], True), s["x"].detach().double().requires_grad_()
    y = _layer_ref(w, "", x)
    y.backward(s["grad"].double())
    return {"y": y.detach(), "x": x.grad, "w": {n: p.grad for n, p in w.items()}}


def _exact_train_step(s):
    w = _double(s["model"], True)
    x = torch.log_softmax(_model_ref(w, s["ids"], s["layers"])[:, :-1], -1)
    lp = x.gather(-1, s["ids"][:, 1:, None])[..., 0]
    loss, adv = _loss_ref(lp, s, s["old"][:, 1:], s["mask"][:, 1:])
    loss.backward()
    return {"loss": loss.detach(), "lp": lp.detach(), "adv": adv, "w": {n: p.grad for n, p in w.items()}}
