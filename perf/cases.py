"""The calls whose time this repository watches: what a QLoRA training run of a Qwen2-shaped model
asks of the framework, from one small weight expansion to the whole training step, with the exact
(64-bit) answer of each and the error another correct implementation may have.

Every case goes through the package's public entry points. `graph` marks the calls captured in a HIP
graph, as the framework's own GraphedStep / BucketedGraphSteps run every layer of a training step;
the others are issued eagerly.
"""

import math

import torch

from claudemaxing_amd import lm_head_loss, qlora_step
from claudemaxing_amd.attention import packed_causal_attention
from claudemaxing_amd.nf4 import QuantState, dequantize_nf4, dynamic_code_map
from claudemaxing_amd.qkv import fused_qkv
from claudemaxing_amd.rmsnorm import add_norm, norm_pass, rmsnorm
from claudemaxing_amd.rope import rope
from claudemaxing_amd.swiglu_recompute import swiglu_recompute

DEVICE = "cuda"
HEAD_DIM = 128
EPS = 1e-6
THETA = 1e6
VOCAB = 151936
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SIZE = {"fp16": 2, "bf16": 2, "fp32": 4}

# (hidden, ffn, query heads, key/value heads): the decoder shapes of the step's configuration and of
# the tests of the other model sizes
SHAPES = ((1536, 8960, 12, 2), (2048, 11008, 16, 2), (3584, 18944, 28, 4))


def listed():
    return [
        # the smallest expansion of a training step (k_proj), and of the calls in general: a
        # bitsandbytes-style layer asks for it once per forward and once per backward
        {"name": "dequant_k", "kind": "dequant", "rows": 256, "cols": 1536, "dtype": "fp16",
         "blocksize": 64, "nested": True},
        # gate_proj of the 1536-wide model: the expansion the reference publishes a time for
        {"name": "dequant_gate", "kind": "dequant", "rows": 8960, "cols": 1536, "dtype": "fp16",
         "blocksize": 64, "nested": True},
        # the norm and the rotary embedding of one layer, forward and backward, called one by one
        # on a packed batch of 4 rows of 128..512 tokens
        {"name": "norm_rope_1193", "kind": "norm_rope", "tokens": 1193, "hidden": 1536,
         "heads": 12, "kv": 2, "dtype": "fp16"},
        # the MLP activation of a full 4 x 512 batch, both directions
        {"name": "swiglu_2048", "kind": "swiglu", "tokens": 2048, "ffn": 8960, "dtype": "fp16"},
        # a layer's input norm and q/k/v projections with their adapters, both directions, at the
        # token count of the benchmark's fixed batch, inside a captured step
        {"name": "qkv_1276", "kind": "qkv", "tokens": 1276, "hidden": 1536, "ffn": 8960,
         "heads": 12, "kv": 2, "graph": True},
        # its attention over the same batch's four rows, and one long document
        {"name": "attn_1276", "kind": "attn", "rows": "154,284,482,356", "heads": 12, "kv": 2,
         "graph": True},
        {"name": "attn_8191", "kind": "attn", "rows": "8191", "heads": 12, "kv": 2,
         "graph": False},
        # its second norm and MLP at that token count, and on a batch of long documents
        {"name": "mlp_1276", "kind": "mlp", "tokens": 1276, "hidden": 1536, "ffn": 8960,
         "heads": 12, "kv": 2, "graph": True},
        {"name": "mlp_8192", "kind": "mlp", "tokens": 8192, "hidden": 1536, "ffn": 8960,
         "heads": 12, "kv": 2, "graph": False},
        # the head and loss of one short example, and of a full 4 x 512 batch
        {"name": "head_131", "kind": "head", "tokens": 131, "vocab": VOCAB, "hidden": 1536,
         "dtype": "fp16", "grad": True},
        {"name": "head_2048", "kind": "head", "tokens": 2048, "vocab": VOCAB, "hidden": 1536,
         "dtype": "fp16", "grad": True},
        # the whole training step of the 28-layer model, replayed from its graph, with the
        # optimizer
        {"name": "step_graphed", "kind": "step", "layers": 28, "lengths": 1, "graph": True},
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    hidden, ffn, heads, kv = rng.choice(SHAPES[:1] * 2 + SHAPES)
    kind = rng.choice(("dequant", "norm_rope", "swiglu", "qkv", "attn", "mlp", "head") * 2
                      + ("step",))
    if kind == "dequant":
        rows, cols = rng.choice(((kv * HEAD_DIM, hidden), (heads * HEAD_DIM, hidden),
                                 (ffn, hidden), (hidden, ffn), (64 * log(1, 128), 64 * log(1, 64))))
        return {"kind": kind, "rows": rows, "cols": cols,
                "dtype": rng.choice(("fp16", "fp16", "bf16", "fp32")),
                "blocksize": rng.choice((64, 64, 128)), "nested": rng.random() < 0.8}
    if kind == "norm_rope":
        return {"kind": kind, "tokens": log(33, 32768), "hidden": hidden, "heads": heads, "kv": kv,
                "dtype": rng.choice(("fp16", "fp16", "bf16", "fp32"))}
    if kind == "swiglu":
        return {"kind": kind, "tokens": log(33, 8192), "ffn": ffn,
                "dtype": rng.choice(("fp16", "fp16", "bf16"))}
    if kind == "qkv":  # the adapters' fused path: inputs of up to 2048 columns
        hidden, ffn, heads, kv = rng.choice(SHAPES[:1] * 2 + SHAPES[:2])
        tokens = log(65, 8192)
        return {"kind": kind, "tokens": tokens, "hidden": hidden, "ffn": ffn, "heads": heads,
                "kv": kv, "graph": tokens < 3000}
    if kind == "attn":
        if rng.random() < 0.5:  # a batch of short rows
            rows = [rng.randint(64, 512) for _ in range(rng.choice((2, 4, 8, 16)))]
        else:  # one to three long documents
            rows = [log(512, 8192) for _ in range(rng.randint(1, 3))]
            while sum(rows) > 8191:
                rows[rows.index(max(rows))] = max(rows) * 2 // 3
        return {"kind": kind, "rows": ",".join(map(str, rows)), "heads": heads, "kv": kv,
                "graph": sum(rows) < 3000}
    if kind == "mlp":
        tokens = log(65, 8192 * 8960 // ffn * 1536 // hidden)
        return {"kind": kind, "tokens": tokens, "hidden": hidden, "ffn": ffn, "heads": heads,
                "kv": kv, "graph": tokens < 3000}
    if kind == "head":
        return {"kind": kind, "tokens": log(65, 4096), "vocab": VOCAB, "hidden": hidden,
                "dtype": rng.choice(("fp16", "fp16", "fp16", "bf16")),
                "grad": rng.random() < 0.75}
    return {"kind": kind, "layers": rng.randint(2, 6), "lengths": rng.randint(2, 999),
            "graph": rng.random() < 0.67}


# -- inputs --------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(DEVICE).manual_seed(1000003 * seed + 17)


def _normal(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEVICE) * std).to(dtype)


def _quantized(case, seed):
    """N(0, 0.02) weights in the 4-bit layout, as plain tensors: (packed, absmax, absmax2, code2,
    offset); without double quantization absmax is fp32 and the rest None."""
    g = _generator(seed)
    bs = case["blocksize"]
    w = _normal(g, case["rows"] * case["cols"] // bs, bs, std=0.02)
    absmax = w.abs().amax(1)
    code = _code()
    idx = torch.bucketize(w / absmax[:, None], (code[1:] + code[:-1]) / 2).to(torch.uint8)
    idx = idx.reshape(-1, 2)
    packed = ((idx[:, 0] << 4) | idx[:, 1]).reshape(-1, 1).contiguous()
    if not case["nested"]:
        return packed, absmax, None, None, None
    offset = absmax.mean()
    centred = absmax - offset
    pad = (-centred.numel()) % 256
    blocks = torch.cat([centred, centred.new_zeros(pad)]).reshape(-1, 256)
    absmax2 = blocks.abs().amax(1)
    code2 = dynamic_code_map().to(DEVICE)
    q8 = torch.bucketize(blocks / absmax2[:, None], (code2[1:] + code2[:-1]) / 2)
    q8 = q8.reshape(-1)[:centred.numel()].to(torch.uint8).contiguous()
    return packed, q8, absmax2, code2, offset


def _code():
    """The NF4 code table (QLoRA, arXiv:2305.14314, Appendix E)."""
    return torch.tensor((
        -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
        -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
        0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
        0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0), device=DEVICE)


def _expanded(packed, absmax, absmax2, code2, offset, blocksize, blocksize2=256):
    """The fp32 values of a 4-bit weight [blocks, blocksize], in plain torch."""
    if absmax2 is not None:
        second = absmax2.repeat_interleave(blocksize2)[:absmax.numel()]
        absmax = code2[absmax.long()] * second + offset
    b = packed.reshape(-1).long()
    values = _code()[torch.stack([b >> 4, b & 15], 1)]
    return values.reshape(-1, blocksize) * absmax[:, None]


def _dense(linear):
    """The fp16 weight an NF4 layer holds, in 64 bits."""
    s = linear.quant_state
    w = _expanded(linear.packed, s.absmax, s.state2.absmax, s.state2.code, s.offset, s.blocksize)
    return w.to(torch.float16).double().reshape(tuple(s.shape))


def _tables(lengths):
    """Rotary cos and sin of packed rows, [1, N, 128] fp32."""
    pos = torch.cat([torch.arange(n) for n in lengths]).to(DEVICE).float()
    inv = THETA ** (-torch.arange(0, HEAD_DIM, 2, device=DEVICE).float() / HEAD_DIM)
    angle = (pos[:, None] * inv[None, :]).repeat(1, 2)
    return angle.cos()[None].contiguous(), angle.sin()[None].contiguous()


def _layer(case, seed):
    """One decoder layer of the QLoRA model of this shape, its adapters away from their start (a
    zero lora_B would leave lora_A without a gradient)."""
    lm = qlora_step.build_model(
        DEVICE, seed=seed, num_hidden_layers=1, vocab_size=64, hidden_size=case["hidden"],
        intermediate_size=case["ffn"], num_attention_heads=case["heads"],
        num_key_value_heads=case["kv"])
    _move_adapters(lm, seed)
    layer = lm.model.layers[0]
    g = _generator(seed + 5)
    with torch.no_grad():
        for norm in (layer.input_layernorm, layer.post_attention_layernorm):
            norm.weight.copy_(torch.rand(case["hidden"], generator=g, device=DEVICE) + 0.5)
    return layer


def _move_adapters(lm, seed):
    g = _generator(seed + 3)
    with torch.no_grad():
        for name, p in lm.named_parameters():
            if "lora_B" in name:
                p.copy_(_normal(g, *p.shape, std=0.01))


def _norm_weight(g, hidden):
    """Norm weights in [0.5, 1.5] with a twentieth of the channels nearly off."""
    w = torch.rand(hidden, generator=g, device=DEVICE) + 0.5
    off = torch.rand(hidden, generator=g, device=DEVICE) < 0.05
    return torch.where(off, torch.full_like(w, 1e-4), w)


def _head_inputs(case, seed):
    g = _generator(seed)
    dt = DTYPES[case["dtype"]]
    weight = _normal(g, case["vocab"], case["hidden"], dtype=dt, std=0.02)
    tokens = case["tokens"]
    target = torch.randint(0, case["vocab"], (1, tokens), generator=g, device=DEVICE)
    # hidden states that lean on their label's row by a random amount: from tokens the model has
    # no idea of to tokens it is sure of
    lean = torch.rand(tokens, 1, generator=g, device=DEVICE) * 25
    hidden = _normal(g, tokens, case["hidden"]) + lean * weight[target[0]].float()
    ignored = torch.rand(1, tokens, generator=g, device=DEVICE) < 0.1
    return hidden.to(dt)[None], weight, torch.where(ignored, -100, target)


def _inputs(case, seed):
    """The tensors of a case, made from the seed."""
    kind = case["kind"]
    if kind == "dequant":
        return _quantized(case, seed)
    if kind == "head":
        return _head_inputs(case, seed)
    g = _generator(seed)
    if kind == "norm_rope":
        n, h, dt = case["tokens"], case["hidden"], DTYPES[case["dtype"]]
        x, dy = _normal(g, n, h, dtype=dt), _normal(g, n, h, dtype=dt)
        weight = _norm_weight(g, h).to(dt)
        qk = [_normal(g, 1, n, heads, HEAD_DIM, dtype=dt).transpose(1, 2)
              for heads in (case["heads"], case["kv"])]
        grads = [_normal(g, 1, heads, n, HEAD_DIM, dtype=dt)
                 for heads in (case["heads"], case["kv"])]
        cos, sin = _tables(_row_lengths(n))
        return x, weight, dy, *qk, cos.to(dt), sin.to(dt), *grads
    if kind == "swiglu":
        return tuple(_normal(g, case["tokens"], case["ffn"], dtype=DTYPES[case["dtype"]])
                     for _ in range(3))
    if kind == "attn":
        lengths = [int(n) for n in case["rows"].split(",")]
        n, heads, kv = sum(lengths), case["heads"], case["kv"]
        q = _normal(g, 1, n, heads, HEAD_DIM)  # q and v in the residual stream's fp32, as the
        k = _normal(g, 1, n, kv, HEAD_DIM, dtype=torch.float16)  # projections hand them over
        v = _normal(g, 1, n, kv, HEAD_DIM)
        dout = _normal(g, 1, n, heads, HEAD_DIM, dtype=torch.float16)
        return (*(t.transpose(1, 2) for t in (q, k, v)), dout, *_tables(lengths))
    n, h = case["tokens"], case["hidden"]
    stream = _normal(g, 1, n, h)
    if kind == "qkv":
        kvd = case["kv"] * HEAD_DIM
        return (stream, _normal(g, 1, n, case["heads"] * HEAD_DIM),
                _normal(g, 1, n, kvd, dtype=torch.float16), _normal(g, 1, n, kvd),
                _normal(g, 1, n, h))
    return stream, _normal(g, 1, n, h, std=0.3), _normal(g, 1, n, h)  # mlp


def _row_lengths(n):
    """A packed batch of n tokens in rows of at most 512."""
    full, rest = divmod(n, 512)
    return [512] * full + ([rest] if rest else [])


# -- one pass ------------------------------------------------------------------------------------
_SIDE = []


def _side_stream():
    """One stream for every capture: torch keeps a BLAS workspace per stream."""
    if not _SIDE:
        _SIDE.append(torch.cuda.Stream())
    return _SIDE[0]


class _Call:
    """The state of a case: `body()` is one pass; captured, a pass replays it."""

    def __init__(self, body, graph=False, seed=None):
        self.body, self.seed, self.graph = body, seed, None
        if not graph:
            return
        side = _side_stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            body()
        torch.cuda.current_stream().wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=side):
            self.out = body()

    def __call__(self):
        if self.seed is not None:  # the dropout masks of this pass
            torch.cuda.default_generators[torch.cuda.current_device()].manual_seed(self.seed)
        if self.graph is None:
            return self.body()
        self.graph.replay()
        return self.out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed)
    x = _inputs(case, seed)
    if kind == "dequant":
        return _prepare_dequant(case, x)
    if kind == "norm_rope":
        return _Call(lambda: _norm_rope(*x))
    if kind == "swiglu":
        return _Call(lambda: _swiglu(*x))
    if kind == "attn":
        bounds = [0]
        for n in case["rows"].split(","):
            bounds.append(bounds[-1] + int(n))
        return _Call(lambda: _attention(tuple(bounds), *x), case["graph"])
    if kind == "head":
        return _Call(lambda: _head(case, *x))
    layer = _layer(case, seed)
    if kind == "qkv":
        return _Call(lambda: _qkv(layer, *x), case["graph"], seed)
    return _Call(lambda: _mlp(layer, *x), case["graph"])


def run(state):
    return state()


def _prepare_dequant(case, x):
    packed, absmax, absmax2, code2, offset = x
    second = None
    if case["nested"]:
        second = QuantState(absmax=absmax2, code=code2, blocksize=256, dtype=torch.float32)
    dt = DTYPES[case["dtype"]]
    state = QuantState(absmax=absmax, shape=torch.Size((case["rows"], case["cols"])),
                       code=_code(), blocksize=case["blocksize"], dtype=dt, offset=offset,
                       state2=second)
    return _Call(lambda: dequantize_nf4(packed, state, dt))


def _leaf(t):
    return t.detach().requires_grad_()


def _norm_rope(x, weight, dy, q, k, cos, sin, gq, gk):
    x, q, k = _leaf(x), _leaf(q), _leaf(k)
    out = rmsnorm(x, weight, EPS)
    rq, rk = rope(q, k, cos, sin)
    return (out, rq, rk, *torch.autograd.grad((out, rq, rk), (x, q, k), (dy, gq, gk)))


def _swiglu(gate, up, grad):
    g, u = _leaf(gate), _leaf(up)
    out = swiglu_recompute(g, u)
    return (out, *torch.autograd.grad(out, (g, u), grad))


def _attention(bounds, q, k, v, dout, cos, sin):
    q, k, v = _leaf(q), _leaf(k), _leaf(v)
    out = packed_causal_attention(q, k, v, bounds, cos=cos, sin=sin)
    return (out, *torch.autograd.grad(out, (q, k, v), dout))


def _qkv(layer, hidden, gq, gk, gv, gpass):
    attn, norm = layer.self_attn, layer.input_layernorm
    hidden = _leaf(hidden)
    adapters = [p for m in (attn.q_proj, attn.v_proj) for p in (m.lora_A.weight, m.lora_B.weight)]
    with torch.autocast("cuda", dtype=torch.float16):
        y, residual = norm_pass(hidden, norm.weight, norm.variance_epsilon)
        q, k, v = fused_qkv(attn, y)
    grads = torch.autograd.grad((q, k, v, residual), (hidden, *adapters), (gq, gk, gv, gpass))
    return (q, k, v, *grads)


def _mlp(layer, residual, attn, grad):
    norm = layer.post_attention_layernorm
    residual, attn = _leaf(residual), _leaf(attn)
    with torch.autocast("cuda", dtype=torch.float16):
        y, h = add_norm(residual, attn, norm.weight, norm.variance_epsilon)
        out = layer.mlp(y, residual=h)
    return (out, *torch.autograd.grad(out, (residual, attn), grad))


def _head(case, hidden, weight, target):
    if not case["grad"]:
        with torch.no_grad():
            loss, terms = lm_head_loss.fused_head_loss(hidden, weight, None, target=target)
        return loss, terms.token_loss, terms.token_entropy, terms.correct, terms.labelled
    hidden = _leaf(hidden)
    loss, terms = lm_head_loss.fused_head_loss(hidden, weight, None, target=target)
    (g,) = torch.autograd.grad(loss, hidden)
    return loss, terms.token_loss, terms.token_entropy, terms.correct, terms.labelled, g


def _prepare_step(case, seed):
    lm = qlora_step.build_model(DEVICE, seed=seed, num_hidden_layers=case["layers"])
    _move_adapters(lm, seed)
    opt = qlora_step.make_optimizer(lm)
    scaler = torch.amp.GradScaler("cuda")
    _, lengths = qlora_step.make_batch("cpu", seed=case["lengths"])
    batch, _ = qlora_step.make_batch(DEVICE, seed=case["lengths"])
    g = _generator(seed)
    ids = torch.randint(0, VOCAB, batch["input_ids"].shape, generator=g, device=DEVICE)
    ids = ids * batch["attention_mask"]
    batch.update(input_ids=ids, labels=torch.where(batch["attention_mask"].bool(), ids, -100))
    params = qlora_step.lora_parameters(lm)
    per_layer = len(params) // case["layers"]

    def outputs(loss, metrics):
        # the updated adapters, one output per kind of weight
        weights = [torch.stack([p.detach() for p in params[i::per_layer]])
                   for i in range(per_layer)]
        return [loss, metrics["entropy"], metrics["num_tokens"], *weights]

    if not case["graph"]:
        def eager():
            metrics = {}
            loss = qlora_step.train_step(lm, opt, scaler, batch, metrics=metrics)
            return outputs(loss, metrics)

        return _Call(eager, seed=seed)
    step = qlora_step.GraphedStep(lm, opt, scaler, batch)

    def graphed():
        metrics = {}
        loss = step.step(metrics, batch)
        terms = [t.clone() for t in (step.terms.token_loss, step.terms.token_entropy)]
        grads = [torch.stack(step.grads[i::per_layer]) for i in range(per_layer)]
        return outputs(loss, metrics) + terms + grads

    return _Call(graphed, seed=seed)


# -- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "dequant":
        n = case["rows"] * case["cols"]
        scales = n / case["blocksize"]
        scales = scales + 4 * scales / 256 + 1024 if case["nested"] else 4 * scales
        return {"bytes": n / 2 + scales + n * SIZE[case["dtype"]], "flops": n}
    if kind == "norm_rope":
        n, s = case["tokens"], SIZE[case["dtype"]]
        width = (case["heads"] + case["kv"]) * HEAD_DIM
        norm = 5 * s * n * case["hidden"]  # x, out; dy, x, dx
        rot = 4 * s * n * width + 2 * s * n * HEAD_DIM  # in and out, both ways; the tables
        return {"bytes": norm + rot, "flops": 12 * n * case["hidden"] + 12 * n * width}
    if kind == "swiglu":
        n = case["tokens"] * case["ffn"]  # gate, up, out; grad, d_gate, d_up
        return {"bytes": 6 * SIZE[case["dtype"]] * n, "flops": 20 * n}
    if kind == "attn":
        lengths = [int(n) for n in case["rows"].split(",")]
        n, heads, kv = sum(lengths), case["heads"], case["kv"]
        pairs = sum(m * (m + 1) // 2 for m in lengths)
        moved = n * HEAD_DIM * (heads * (4 + 2 + 2 + 4) + kv * (2 + 4 + 2 + 4) + 2 * 4)
        return {"bytes": moved, "flops": 14 * pairs * HEAD_DIM * heads}
    if kind == "head":
        n, h, v, s = case["tokens"], case["hidden"], case["vocab"], SIZE[case["dtype"]]
        both = 2 if case["grad"] else 1
        return {"bytes": v * h * s + both * n * h * s + 20 * n, "flops": both * 2 * n * v * h}
    if kind == "step":
        _, lengths = qlora_step.make_batch("cpu", seed=case["lengths"])
        lengths = lengths.tolist()
        h, f, heads, kv = SHAPES[0]
        n, layers = sum(lengths), case["layers"]
        rows = ",".join(map(str, lengths))
        shape = {"tokens": n, "hidden": h, "ffn": f, "heads": heads, "kv": kv}
        total = {"bytes": 0, "flops": 0}
        parts = [(layers, dict(shape, kind="qkv")), (layers, dict(shape, kind="mlp")),
                 (layers, dict(kind="attn", rows=rows, heads=heads, kv=kv)),
                 (1, dict(kind="head", tokens=n, hidden=h, vocab=VOCAB, dtype="fp16", grad=True))]
        for times, part in parts:
            w = work(part)
            total = {k: total[k] + times * w[k] for k in total}
        o = heads * HEAD_DIM * h  # the output projection, forward and input gradient
        return {"bytes": total["bytes"] + layers * (o / 2 + n * heads * HEAD_DIM * 4 + n * h * 8),
                "flops": total["flops"] + layers * 4 * n * o}
    n, h, f = case["tokens"], case["hidden"], case["ffn"]
    if kind == "qkv":
        out = (case["heads"] + 2 * case["kv"]) * HEAD_DIM
        # the stream, its two gradients; q, k, v and theirs; the packed weights
        moved = 12 * n * h + 2 * n * HEAD_DIM * (4 * case["heads"] + 6 * case["kv"]) + h * out / 2
        adapters = 16 * (2 * h + (case["heads"] + case["kv"]) * HEAD_DIM)
        return {"bytes": moved + 8 * adapters, "flops": n * (4 * h * out + 6 * adapters)}
    # mlp: the stream, the attention output, the result, its gradient and theirs; the weights;
    # three products each way (the recomputation of gate and up is the implementation's own choice)
    return {"bytes": 24 * n * h + 3 * h * f / 2, "flops": 12 * n * h * f}


# -- what it may be off by -----------------------------------------------------------------------
def tolerance(case):
    """About four times what each kind of call was measured to be off the 64-bit answer."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind in ("norm_rope", "swiglu"):
        # one or two roundings to the data type at the end of fp32 arithmetic
        return {"rel": {"fp16": 1.2e-3, "bf16": 9e-3, "fp32": 3e-7}[case["dtype"]]}
    if kind == "attn":
        return {"rel": 2e-3}  # fp16 operands and probabilities, fp32 sums
    if kind == "head":
        # 16-bit logits; the gradient through 16-bit probabilities, the sure tokens' the worst
        return {"rel": 8e-3 if case["dtype"] == "fp16" else 1.4e-2}
    if kind == "step":
        # an fp16 rounding travels through every layer: between the two ways this package has of
        # multiplying by a 4-bit weight, 5e-3 in the gradients after three steps (one value by 0.1)
        return {"rel": 2e-2, "max": 0.4}
    return {"rel": 2e-3}  # fp16 operands and intermediates, fp32 sums


# -- the answer in 64 bits -----------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None
    if kind in ("qkv", "mlp"):
        layer = _layer(case, seed)
    x = _inputs(case, seed)
    with torch.no_grad():
        if kind == "dequant":
            return _expanded(*x, case["blocksize"]).double().reshape(case["rows"], case["cols"])
        if kind == "norm_rope":
            return _exact_norm_rope(*(t.double() for t in x))
        if kind == "swiglu":
            return _exact_swiglu(*(t.double() for t in x))
        if kind == "attn":
            return _exact_attention([int(n) for n in case["rows"].split(",")],
                                    *(t.double() for t in x))
        if kind == "head":
            return _exact_head(case["grad"], *x)
        if kind == "qkv":
            return _exact_qkv(layer, seed, *x)
        return _exact_mlp(layer, *(t.double() for t in x))


def _rms(x, w):
    r = (x.square().mean(-1, keepdim=True) + EPS).rsqrt()
    return x * r * w, r


def _rms_grad(x, w, r, dy):
    g = dy * w
    return r * (g - x * r.square() * (g * x).mean(-1, keepdim=True))


def _rotate(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat([-b, a], -1) * sin


def _rotate_back(g, cos, sin):
    a, b = (g * sin).chunk(2, -1)
    return g * cos + torch.cat([b, -a], -1)


def _exact_norm_rope(x, w, dy, q, k, cos, sin, gq, gk):
    out, r = _rms(x, w)
    c, s = cos[:, None], sin[:, None]
    return (out, _rotate(q, c, s), _rotate(k, c, s), _rms_grad(x, w, r, dy),
            _rotate_back(gq, c, s), _rotate_back(gk, c, s))


def _silu_grads(gate, up, grad):
    sig = torch.sigmoid(gate)
    return grad * up * sig * (1 + gate * (1 - sig)), grad * gate * sig


def _exact_swiglu(gate, up, grad):
    return (gate * torch.sigmoid(gate) * up, *_silu_grads(gate, up, grad))


def _exact_attention(lengths, q, k, v, dout, cos, sin):
    c, s = cos[:, None], sin[:, None]
    scale = HEAD_DIM ** -0.5
    qr, kr = _rotate(q, c, s), _rotate(k, c, s)
    out, dq, dk, dv = dout.clone(), qr.clone(), torch.zeros_like(kr), torch.zeros_like(v)
    per = q.shape[1] // k.shape[1]
    at = 0
    for n in lengths:
        e = at + n
        future = torch.ones(n, n, dtype=torch.bool, device=DEVICE).triu(1)
        for h in range(q.shape[1]):
            qh, kh, vh = qr[0, h, at:e], kr[0, h // per, at:e], v[0, h // per, at:e]
            p = torch.softmax((qh @ kh.t() * scale).masked_fill_(future, -math.inf), -1)
            o = p @ vh
            do = dout[0, at:e, h]
            out[0, at:e, h] = o
            ds = p * (do @ vh.t() - (do * o).sum(-1, keepdim=True)) * scale
            dq[0, h, at:e] = ds @ kh
            dk[0, h // per, at:e] += ds.t() @ qh
            dv[0, h // per, at:e] += p.t() @ do
        at = e
    return out, _rotate_back(dq, c, s), _rotate_back(dk, c, s), dv


def _exact_head(want_grad, hidden, weight, target):
    h, tgt = hidden[0].double(), target[0]
    labelled = tgt != -100
    losses, entropies, grads, correct = [], [], [], 0
    for i in range(0, h.shape[0], 256):  # rows at a time: the logits are 311 MB per 256
        rows, t, ok = h[i:i + 256], tgt[i:i + 256].clamp(min=0), labelled[i:i + 256]
        z = torch.cat([rows @ weight[j:j + 16384].double().t()
                       for j in range(0, weight.shape[0], 16384)], 1)
        lse = z.logsumexp(1)
        zt = z.gather(1, t[:, None])[:, 0]
        correct += int(((z.argmax(1) == t) & ok).sum())
        losses.append(torch.where(ok, lse - zt, 0.0))
        p = torch.softmax(z, 1)
        entropies.append(lse - (p * z).sum(1))
        if want_grad:
            p.scatter_add_(1, t[:, None], -torch.ones_like(t, dtype=p.dtype)[:, None])
            p *= ok[:, None]
            grads.append(sum(p[:, j:j + 16384] @ weight[j:j + 16384].double()
                             for j in range(0, weight.shape[0], 16384)))
    loss, entropy, n = torch.cat(losses), torch.cat(entropies), int(labelled.sum())
    out = (loss.sum() / n, loss[None], entropy[None], correct, n)
    return (*out, torch.cat(grads)[None] / n) if want_grad else out


def _exact_qkv(layer, seed, hidden, gq, gk, gv, gpass):
    attn = layer.self_attn
    w = layer.input_layernorm.weight.double()
    x = hidden.double()
    y, r = _rms(x, w)
    torch.cuda.default_generators[torch.cuda.current_device()].manual_seed(seed)
    outs, dy, adapters = [], torch.zeros_like(y), []
    for name, g in (("q_proj", gq), ("k_proj", gk), ("v_proj", gv)):
        m, g = getattr(attn, name), g.double()
        base = m if name == "k_proj" else m.base_layer
        dense = _dense(base)
        out = y @ dense.t() + base.bias.double()
        dy += g @ dense
        if name != "k_proj":
            a, b, s = m.lora_A.weight.double(), m.lora_B.weight.double(), m.scaling
            keep = torch.native_dropout(hidden, m.p, True)[1].double() / (1 - m.p)
            xd = y * keep
            ax = xd @ a.t()
            out += ax @ b.t() * s
            ga = g @ b * s
            dy += (ga @ a) * keep
            adapters += [ga[0].t() @ xd[0], g[0].t() @ ax[0] * s]
        outs.append(out)
    return (*outs, _rms_grad(x, w, r, dy) + gpass.double(), *adapters)


def _exact_mlp(layer, residual, attn, grad):
    m, w = layer.mlp, layer.post_attention_layernorm.weight.double()
    h = residual + attn
    y, r = _rms(h, w)
    wg, wu, wd = (_dense(p) for p in (m.gate_proj, m.up_proj, m.down_proj))
    gate, up = y @ wg.t(), y @ wu.t()
    out = h + (gate * torch.sigmoid(gate) * up) @ wd.t()
    dg, du = _silu_grads(gate, up, grad @ wd)
    dh = grad + _rms_grad(h, w, r, dg @ wg + du @ wu)
    return out, dh, dh
