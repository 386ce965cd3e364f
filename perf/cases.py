"""What the speed of this framework is measured on.

Each case is one kind of call that a user's program makes through the public
entry points, at sizes of the repository's own workloads (BERT-base and the
Qwen3-VL-2B-shaped text tower: hidden 768 / 3072 and 2048 / 6144, LoRA rank 16
and 32, one scale per row or per group of 64) and at ragged sizes between.

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same
ranges; ``prepare`` makes what a program holds before the call, ``run`` is one
pass, ``exact`` the same result in float64 by plain torch.

Kinds:

* ``infer``   one INT4 + LoRA projection, no gradients, bf16 (queries and
  small batches at serving time: 1 to 2048 rows);
* ``shared``  the q / k / v projections of one input, no gradients (1 to 64
  rows);
* ``query``   a Qwen3-wide layer's forward over one short query, no
  gradients, captured in a graph as a serving loop keeps it;
* ``linear``  one INT4 + LoRA projection, forward and backward: bf16, float32
  (the default ``PrecisionConfig``) or no policy (bf16 activations against
  the float32 masters);
* ``gelu`` / ``swiglu``  the feed-forward blocks, forward and backward;
* ``fp8``     the fp8 ``Linear`` with its fp32 master weight, forward and
  backward, dynamic scaling or delayed scaling with its per-step update;
* ``bert`` / ``qwen3``  one whole encoder layer, forward and backward;
* ``step``    a captured train step (forward, rematerialized backward,
  clipping and AdamW) of a two-layer BERT-base-wide encoder.
"""

from __future__ import annotations

import math
from contextlib import nullcontext

import torch
import torch.nn.functional as F

from representax_amd import (FP32_POLICY, DelayedScaling, Linear, PrecisionConfig, QuantizedLoRALinear,
                             gelu_mlp, model_for_compute, precision_context,
                             resolve_precision_policy, shared_input_projections, swiglu_mlp)
from representax_amd.trainstep import (BertConfig, MNRTrainStep, Qwen3TextConfig,
                                       build_int4lora_encoder, build_int4lora_qwen3)

DEVICE = "cuda"
BF16 = torch.bfloat16
F64 = torch.float64
POLICY = resolve_precision_policy(PrecisionConfig.bfloat16_mixed())
VOCABULARY = 2048  # rows of the harnesses' embedding tables (not on the measured path)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one query's single token row through a Qwen3-wide FFN projection: the
        # smallest call, where launches and latency count
        {"name": "infer_m1_2048x6144", "kind": "infer", "m": 1, "k": 2048, "n": 6144, "rank": 32,
         "group": 64, "bias": False},
        # one query of 13 tokens through a Qwen3-wide layer, replayed
        {"name": "query_qwen3_1x13", "kind": "query", "batch": 1, "sequence": 13, "rank": 32,
         "group": 64},
        # a few short queries packed together, between the small-row kernels
        # and the training sizes
        {"name": "infer_m333_2048x6144", "kind": "infer", "m": 333, "k": 2048, "n": 6144,
         "rank": 32, "group": 64, "bias": False},
        # one BERT-base FFN up projection of 32 sequences of 128 tokens, the
        # reference's own scale layout (one per row), with its bias
        {"name": "linear_4096_768x3072", "kind": "linear", "m": 4096, "k": 768, "n": 3072,
         "rank": 16, "group": 0, "bias": True, "precision": "bfloat16"},
        # the same projection under the default float32 precision, 8 sequences
        # of 125 tokens
        {"name": "linear_f32_1000_768x3072", "kind": "linear", "m": 1000, "k": 768, "n": 3072,
         "rank": 16, "group": 64, "bias": True, "precision": "float32"},
        # the BERT-base FFN at the train step's 64 pairs of 256 tokens
        {"name": "gelu_32768_768x3072", "kind": "gelu", "m": 32768, "k": 768, "n": 3072,
         "rank": 16, "group": 64},
        # the Qwen3-wide FFN at the train step's 32 sequences of 512 tokens
        {"name": "swiglu_16384_2048x6144", "kind": "swiglu", "m": 16384, "k": 2048, "n": 6144,
         "rank": 32, "group": 64},
        # fp8 linears of BERT-base: 8192 tokens, and 7 sequences of 500 tokens
        # with delayed scaling
        {"name": "fp8_8192_768x3072", "kind": "fp8", "m": 8192, "k": 768, "n": 3072,
         "delayed": False},
        {"name": "fp8_delayed_3500_3072x768", "kind": "fp8", "m": 3500, "k": 3072, "n": 768,
         "delayed": True},
        # whole layers: BERT-base at the train step's 64 pairs of 256 tokens,
        # the Qwen3-wide one with a ragged batch of 7 sequences of 500 tokens
        {"name": "bert_layer_128x256", "kind": "bert", "batch": 128, "sequence": 256, "rank": 16,
         "group": 64},
        {"name": "qwen3_layer_7x500", "kind": "qwen3", "batch": 7, "sequence": 500, "rank": 32,
         "group": 64},
        # the captured train step: 256 pairs of 32 tokens, two layers
        {"name": "step_bert2_256x32", "kind": "step", "batch": 256, "sequence": 32, "layers": 2,
         "rank": 16, "group": 64},
    ]


SHAPES = [(2048, 6144, 32), (6144, 2048, 32), (2048, 2048, 32), (2048, 1024, 32),
          (768, 768, 16), (768, 3072, 16), (3072, 768, 16)]


def _log(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "infer", "shared", "query", "linear", "linear", "gelu",
                       "swiglu", "fp8", "fp8", "bert", "qwen3", "step"])
    group = rng.choice([64, 64, 0])
    if kind in ("infer", "linear"):
        k, n, rank = rng.choice(SHAPES)
        case = {"kind": kind, "k": k, "n": n, "rank": rank, "group": group, "bias": rank == 16}
        if kind == "infer":
            return {**case, "m": _log(rng, 1, 2048)}
        precision = rng.choice(["bfloat16", "bfloat16", "float32", "none"])
        # without bf16 matrices, up to 2048 tokens of the BERT-base FFN's work
        most = 16384 if precision == "bfloat16" else 2048 * 768 * 3072 // (k * n)
        return {**case, "m": _log(rng, 64, most), "precision": precision}
    if kind == "shared":
        k, widths, rank = rng.choice([(2048, "2048,1024,1024", 32), (2048, "6144,6144", 32),
                                      (768, "768,768,768", 16)])
        return {"kind": kind, "m": _log(rng, 1, 64), "k": k, "widths": widths, "rank": rank,
                "group": group}
    if kind == "query":
        return {"kind": kind, "batch": _log(rng, 1, 8), "sequence": _log(rng, 4, 64), "rank": 32,
                "group": group}
    if kind == "gelu":
        return {"kind": kind, "m": _log(rng, 256, 32768), "k": 768, "n": 3072, "rank": 16,
                "group": group}
    if kind == "swiglu":
        return {"kind": kind, "m": _log(rng, 256, 16384), "k": 2048, "n": 6144, "rank": 32,
                "group": group}
    if kind == "fp8":
        k, n = rng.choice([(768, 768), (768, 3072), (3072, 768)])
        return {"kind": kind, "m": _log(rng, 512, 8192), "k": k, "n": n,
                "delayed": rng.choice([False, True])}
    if kind == "bert":
        return {"kind": kind, "batch": _log(rng, 4, 128), "sequence": _log(rng, 32, 256),
                "rank": 16, "group": group}
    if kind == "qwen3":
        return {"kind": kind, "batch": _log(rng, 1, 16), "sequence": _log(rng, 64, 512),
                "rank": 32, "group": group}
    batch = _log(rng, 8, 512)
    return {"kind": kind, "batch": batch, "sequence": _log(rng, 16, min(256, 16384 // batch)),
            "layers": 2, "rank": 16, "group": group}


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device=DEVICE) * scale).to(dtype)


def _adapter(g, k, n, rank, group, bias):
    """A trained adapter over a packed projection: W, A and B ~ N(0, 0.02)."""

    base = Linear(_normal(g, n, k, scale=0.02), _normal(g, n, scale=0.02) if bias else None)
    layer = QuantizedLoRALinear.from_linear(base, rank=rank, alpha=2.0 * rank, key=1,
                                            initialization_scale=0.02, group_size=group or None)
    with torch.no_grad():
        layer.lora_a.copy_(_normal(g, rank, k, scale=0.02))
        layer.lora_b.copy_(_normal(g, n, rank, scale=0.02))
    return layer


def _randomize_adapters(module, g):
    for layer in module.modules():
        if isinstance(layer, QuantizedLoRALinear):
            with torch.no_grad():
                layer.lora_a.copy_(_normal(g, *layer.lora_a.shape, scale=0.02))
                layer.lora_b.copy_(_normal(g, *layer.lora_b.shape, scale=0.02))


def _masters(*modules):
    return [p for mod in modules for layer in mod.modules() if isinstance(layer, QuantizedLoRALinear)
            for p in (layer.lora_a, layer.lora_b)]


def _mlp(g, case):
    k, n, rank, group = case["k"], case["n"], case["rank"], case["group"]
    if case["kind"] == "gelu":
        return [_adapter(g, k, n, rank, group, True), _adapter(g, n, k, rank, group, True)]
    return [_adapter(g, k, n, rank, group, False), _adapter(g, k, n, rank, group, False),
            _adapter(g, n, k, rank, group, False)]


def _layer_model(case, seed):
    if case["kind"] in ("qwen3", "query"):
        config = Qwen3TextConfig(vocab_size=VOCABULARY, num_hidden_layers=1)
        model = build_int4lora_qwen3(config, rank=case["rank"], alpha=2.0 * case["rank"],
                                     group_size=case["group"] or None, seed=seed, device=DEVICE)
    else:
        config = BertConfig(vocab_size=VOCABULARY, num_hidden_layers=case.get("layers", 1))
        model = build_int4lora_encoder(config, rank=case["rank"], alpha=2.0 * case["rank"],
                                       group_size=case["group"] or None, seed=seed, device=DEVICE)
    return config, model


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    state = {"kind": kind}
    if kind == "infer":
        layer = _adapter(g, case["k"], case["n"], case["rank"], case["group"], case["bias"])
        state["masters"] = layer
        state["layer"] = model_for_compute(layer, POLICY)
        state["x"] = _normal(g, case["m"], case["k"], dtype=BF16)
    elif kind == "shared":
        layers = [_adapter(g, case["k"], int(n), case["rank"], case["group"], False)
                  for n in case["widths"].split(",")]
        state["masters"] = layers
        state["layers"] = [model_for_compute(layer, POLICY) for layer in layers]
        state["x"] = _normal(g, case["m"], case["k"], dtype=BF16)
    elif kind == "linear":
        layer = _adapter(g, case["k"], case["n"], case["rank"], case["group"], case["bias"])
        precision = case["precision"]
        state["layers"] = [layer]
        state["policy"] = {"bfloat16": POLICY, "float32": FP32_POLICY, "none": None}[precision]
        x_dtype = torch.float32 if precision == "float32" else BF16
        state["x"] = _normal(g, case["m"], case["k"], dtype=x_dtype).requires_grad_(True)
        state["gy"] = _normal(g, case["m"], case["n"],
                              dtype=BF16 if precision == "bfloat16" else torch.float32)
    elif kind in ("gelu", "swiglu"):
        state["layers"] = _mlp(g, case)
        state["x"] = _normal(g, case["m"], case["k"], dtype=BF16).requires_grad_(True)
        state["gy"] = _normal(g, case["m"], case["k"], dtype=BF16)
    elif kind == "fp8":
        m, k, n = case["m"], case["k"], case["n"]
        state["layer"] = Linear(_normal(g, n, k, scale=0.02))
        x = torch.randn((m, k), generator=g, device=DEVICE)
        outliers = torch.rand((m, k), generator=g, device=DEVICE) < 1e-3
        state["x"] = torch.where(outliers, 50.0 * x, x).to(BF16).requires_grad_(True)
        state["gy"] = _normal(g, m, n, dtype=BF16)
        scaling = None
        if case["delayed"]:
            scaling = DelayedScaling.for_model(state["layer"], device=DEVICE)
        config = PrecisionConfig.float8_mixed("delayed" if case["delayed"] else "dynamic")
        state["policy"] = resolve_precision_policy(config, fp8_state=scaling)
        if case["delayed"]:
            run(state)  # an earlier step: the history then holds this data's maxima
    elif kind == "query":
        _, model = _layer_model(case, seed)
        _randomize_adapters(model.layers[0], g)
        state["masters"] = model.layers[0]
        layer = model_for_compute(model.layers[0], POLICY)
        state["x"] = _normal(g, case["batch"], case["sequence"], 2048, dtype=BF16)
        state["extra"] = model.rotary(case["sequence"])

        def forward():
            with torch.no_grad(), precision_context(POLICY):
                return layer(state["x"], *state["extra"])

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            forward()
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["y"] = forward()
        state["layer"] = layer
    elif kind in ("bert", "qwen3"):
        _, model = _layer_model(case, seed)
        state["layer"] = model.layers[0]
        _randomize_adapters(state["layer"], g)
        width = 2048 if kind == "qwen3" else 768
        shape = (case["batch"], case["sequence"], width)
        state["x"] = _normal(g, *shape, dtype=BF16).requires_grad_(True)
        state["gy"] = _normal(g, *shape, dtype=BF16)
        state["extra"] = model.rotary(case["sequence"]) if kind == "qwen3" else (None,)
    else:
        _, model = _layer_model(case, seed)
        _randomize_adapters(model, g)
        step = MNRTrainStep(model, batch=case["batch"], sequence=case["sequence"], seed=seed)
        # capture() runs two steps; the program starts from its own weights
        masters = step.flat.detach().clone()
        step.capture()
        with torch.no_grad():
            step.flat.copy_(masters)
            for moment in step.optimizer.state[step.flat].values():
                moment.zero_()
        state["step"] = step
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _gradients(y, state, leaves):
    return torch.autograd.grad(y, [state["x"], *leaves], state["gy"])


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad(), precision_context(POLICY):
            return state["layer"](state["x"])
    if kind == "shared":
        with torch.no_grad(), precision_context(POLICY):
            return shared_input_projections(state["x"], state["layers"])
    if kind == "query":
        state["graph"].replay()
        return state["y"]
    if kind == "step":
        step = state["step"]
        loss = step()
        return loss, step.grad_norm, step.flat.grad
    if kind == "fp8":
        policy, layer = state["policy"], state["layer"]
        with precision_context(policy):
            y = layer(state["x"])
        dx, dw = _gradients(y, state, [layer.weight])
        if policy.fp8_state is None:
            return y, dx, dw
        policy.fp8_state.update()
        return y, dx, dw, policy.fp8_state.scales
    if kind == "linear":
        layer = state["layers"][0]
        with precision_context(state["policy"]) if state["policy"] else nullcontext():
            y = layer(state["x"])
        return (y, *_gradients(y, state, _masters(layer)))
    with precision_context(POLICY):
        if kind == "gelu":
            y = gelu_mlp(state["x"], *state["layers"])
            leaves = _masters(*state["layers"])
        elif kind == "swiglu":
            y = swiglu_mlp(state["x"], *state["layers"])
            leaves = _masters(*state["layers"])
        else:
            y = state["layer"](state["x"], *state["extra"])
            leaves = _masters(state["layer"])
    return (y, *_gradients(y, state, leaves))


# ---------------------------------------------------------------------------
# bytes and operations that the path cannot do without
# ---------------------------------------------------------------------------
def _weight_bytes(k, n, rank, group):
    return n * k / 2 + 2 * n * (k // group if group else 1) + 2 * rank * (k + n)


def _linear_work(m, k, n, rank, group, backward, reads=1, sizes=(2, 2)):
    """Bytes and operations of one projection. ``reads`` 0: x is counted by
    another projection of the same input; ``sizes``: bytes of an element of x
    and of y."""

    weight = _weight_bytes(k, n, rank, group)
    sx, sy = sizes
    nbytes = weight + m * (sx * reads * k + sy * n)
    flops = 2.0 * m * (k * n + rank * (k + n))
    if backward:
        # read the gradient and x, write dx and the fp32 adapter gradients
        nbytes += weight + m * (sy * n + sx * reads * 2 * k) + 4 * rank * (k + n)
        flops += 2.0 * m * (k * n + 2 * rank * (k + n))
    return nbytes, flops


def _sum(parts):
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def _layer_parts(kind, tokens, sequence, rank, group, backward=True):
    if kind in ("qwen3", "query"):
        h, f, q, kv = 2048, 6144, 2048, 1024
        shapes = [(h, q), (h, kv), (h, kv), (q, h), (h, f), (h, f), (f, h)]
        attention = 2.0 * tokens * sequence * q  # causal: half of both products
    else:
        h, f = 768, 3072
        shapes = [(h, h)] * 4 + [(h, f), (f, h)]
        attention = 4.0 * tokens * sequence * h
    flops = sum(_linear_work(tokens, k, n, rank, group, backward)[1] for k, n in shapes)
    weights = sum(_weight_bytes(k, n, rank, group) for k, n in shapes)
    if not backward:
        return weights + 4 * tokens * h, flops + attention
    weights = 2 * weights + sum(4 * rank * (k + n) for k, n in shapes)
    # the layer's input, output and their gradients
    return weights + 8 * tokens * h, flops + 3 * attention


def work(case):
    kind, group = case["kind"], case["group"] if "group" in case else 0
    if kind in ("infer", "linear"):
        sizes = {"float32": (4, 4), "none": (2, 4)}.get(case.get("precision"), (2, 2))
        return _sum([_linear_work(case["m"], case["k"], case["n"], case["rank"], group,
                                  kind == "linear", sizes=sizes)])
    if kind == "shared":
        widths = [int(n) for n in case["widths"].split(",")]
        return _sum([_linear_work(case["m"], case["k"], n, case["rank"], group, False, i == 0)
                     for i, n in enumerate(widths)])
    if kind in ("gelu", "swiglu"):
        m, k, n = case["m"], case["k"], case["n"]
        shapes = [(k, n), (n, k)] if kind == "gelu" else [(k, n), (k, n), (n, k)]
        flops = sum(_linear_work(m, a, b, case["rank"], group, True)[1] for a, b in shapes)
        weights = sum(2 * _weight_bytes(a, b, case["rank"], group) + 4 * case["rank"] * (a + b)
                      for a, b in shapes)
        return {"bytes": weights + 8 * m * k, "flops": flops}
    if kind == "fp8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * (3 * m * k + 2 * m * n) + 4 * 2 * n * k, "flops": 6.0 * m * k * n}
    if kind in ("bert", "qwen3", "query"):
        tokens = case["batch"] * case["sequence"]
        nbytes, flops = _layer_parts(kind, tokens, case["sequence"], case["rank"], group,
                                     kind != "query")
        return {"bytes": nbytes, "flops": flops}
    tokens = 2 * case["batch"] * case["sequence"]
    nbytes, flops = _layer_parts("bert", tokens, case["sequence"], case["rank"], group)
    masters = case["layers"] * case["rank"] * (4 * 2 * 768 + 2 * (768 + 3072))
    # AdamW: masters, both moments and the gradient read, the first three written
    return {"bytes": case["layers"] * nbytes + 7 * 4 * masters, "flops": case["layers"] * flops}


# ---------------------------------------------------------------------------
# what is allowed, and the same results in float64
# ---------------------------------------------------------------------------
def tolerance(case):
    # bf16 outputs round at 2^-9 relative, and bf16 intermediates (h, dh, the
    # activations of a block) round once each. About four times the distance
    # from float64 that the paths show.
    if case["kind"] == "step":
        return {"rel": 0.03, "max": 0.9}
    if case["kind"] in ("bert", "qwen3"):
        return {"rel": 0.03, "max": 0.5}
    if case.get("precision") == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.01, "max": 0.2}


def _dequantized(layer):
    """The packed base weight, bf16(q * s), in float64 (plain torch)."""

    packed = layer.packed_weight.to(torch.int32)
    q = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(packed.shape[0], -1)
    q = q[:, :layer.input_size]
    q = torch.where(q < 8, q, q - 16).float()
    scales = layer.scale_bits.view(BF16).float().reshape(packed.shape[0], -1)
    scales = scales.repeat_interleave(layer.input_size // scales.shape[1], dim=1)
    return (q * scales).to(BF16).to(F64)


class _Exact:
    """One INT4 + LoRA projection in float64; the adapters are the compute
    views of the fp32 masters, as the policy defines them (bf16)."""

    def __init__(self, layer, gradients=True, views=BF16):
        self.w = _dequantized(layer)
        self.a = layer.lora_a.detach().to(views).to(F64).requires_grad_(gradients)
        self.b = layer.lora_b.detach().to(views).to(F64).requires_grad_(gradients)
        self.c = layer.alpha / layer.rank
        bits = layer.bias_bits
        self.bias = None if bits is None else bits.view(BF16).to(F64)

    def __call__(self, x):
        y = x @ self.w.t() + (x @ self.a.t()) @ self.b.t() * self.c
        return y if self.bias is None else y + self.bias


def _leaves(*linears):
    return [t for linear in linears for t in (linear.a, linear.b)]


def _attend(q, k, v, scale, causal):
    s = (q @ k.transpose(-1, -2)) * scale
    if causal:
        n = s.shape[-1]
        s = s + torch.full((n, n), float("-inf"), dtype=F64, device=s.device).triu(1)
    return torch.softmax(s, dim=-1) @ v


def _norm(x, module):
    return F.layer_norm(x, x.shape[-1:], module.weight.to(F64), module.bias.to(F64), module.eps)


def _rms(x, module):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + module.eps) * module.weight.to(F64)


def _exact_bert(layer, x, linears):
    query, key, value, output, up, down = linears
    b, s, h = x.shape
    heads, d = layer.attention.heads, layer.attention.head_dim
    q, k, v = (f(x).reshape(b, s, heads, d).transpose(1, 2) for f in (query, key, value))
    out = _attend(q, k, v, 1.0 / math.sqrt(d), False).transpose(1, 2).reshape(b, s, h)
    x = _norm(x + output(out), layer.attention_norm)
    return _norm(x + down(F.gelu(up(x))), layer.output_norm)


def _exact_qwen3(layer, x, cos, sin, linears):
    query, key, value, output, gate, up, down = linears
    att = layer.attention
    b, s, _ = x.shape
    heads, kv, d = att.heads, att.kv_heads, att.head_dim
    cos, sin = cos.to(F64)[:, :, None], sin.to(F64)[:, :, None]

    def rotate(t):
        half = torch.cat((-t[..., d // 2:], t[..., :d // 2]), dim=-1)
        return (t * cos + half * sin).transpose(1, 2)

    n = _rms(x, layer.input_norm)
    q = rotate(_rms(query(n).reshape(b, s, heads, d), att.query_norm))
    k = rotate(_rms(key(n).reshape(b, s, kv, d), att.key_norm))
    v = value(n).reshape(b, s, kv, d).transpose(1, 2)
    k = k.repeat_interleave(heads // kv, dim=1)
    v = v.repeat_interleave(heads // kv, dim=1)
    out = _attend(q, k, v, 1.0 / math.sqrt(d), True).transpose(1, 2).reshape(b, s, heads * d)
    x = x + output(out)
    n = _rms(x, layer.post_attention_norm)
    return x + down(F.silu(gate(n)) * up(n))


def _projections(layer):
    return [m for m in layer.modules() if isinstance(m, QuantizedLoRALinear)]


def _quantized(t, fmt):
    """fp8 values of ``t`` under its own dynamic scale, and the scale (the
    definition: float32 divide, round to nearest even)."""

    dtype, top = (torch.float8_e4m3fn, 448.0) if fmt == "e4m3fn" else (torch.float8_e5m2, 57344.0)
    t = t.float()
    # a tensor divisor: torch divides by a number through its reciprocal
    scale = t.abs().max() / torch.full((), top, device=t.device)
    scale = scale.clamp_min(torch.finfo(torch.float32).tiny)
    return (t / scale).to(dtype).to(F64), scale


def exact(case, seed):
    state = prepare(case, seed) if case["kind"] != "step" else None
    kind = case["kind"]
    if kind == "infer":
        return _Exact(state["masters"], False)(state["x"].to(F64))
    if kind == "shared":
        return [_Exact(m, False)(state["x"].to(F64)) for m in state["masters"]]
    if kind == "fp8":
        left, s_left = _quantized(state["x"].detach(), "e4m3fn")
        right, s_right = _quantized(state["layer"].weight.detach().to(BF16), "e4m3fn")
        grad, s_grad = _quantized(state["gy"], "e5m2")
        out = [left @ right.t() * s_left.to(F64) * s_right.to(F64),
               grad @ right * s_grad.to(F64) * s_right.to(F64),
               grad.t() @ left * s_grad.to(F64) * s_left.to(F64)]
        if case["delayed"]:
            out.append(torch.stack((s_left, s_right, s_grad)).to(F64))
        return out
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "query":
        linears = [_Exact(m, False) for m in _projections(state["masters"])]
        return _exact_qwen3(state["masters"], state["x"].to(F64), *state["extra"], linears)
    x = state["x"].detach().to(F64).requires_grad_(True)
    if kind in ("bert", "qwen3"):
        linears = [_Exact(m) for m in _projections(state["layer"])]
        if kind == "bert":
            y = _exact_bert(state["layer"], x, linears)
        else:
            y = _exact_qwen3(state["layer"], x, *state["extra"], linears)
    elif kind == "linear":
        views = BF16 if case["precision"] == "bfloat16" else torch.float32
        linears = [_Exact(state["layers"][0], views=views)]
        y = linears[0](x)
    else:
        linears = [_Exact(m) for m in state["layers"]]
        if kind == "gelu":
            y = linears[1](F.gelu(linears[0](x)))
        else:
            y = linears[2](F.silu(linears[0](x)) * linears[1](x))
    grads = torch.autograd.grad(y, [x, *_leaves(*linears)], state["gy"].to(F64))
    return [y.detach(), *grads]


def _exact_step(case, seed):
    config, model = _layer_model(case, seed)
    _randomize_adapters(model, _generator(seed))
    step = MNRTrainStep(model, batch=case["batch"], sequence=case["sequence"], seed=seed)
    ids = torch.cat([step.query_ids, step.document_ids], 0)
    hidden = (model.word[ids] + model.position[:ids.shape[1]][None]
              + model.token_type[torch.zeros_like(ids)]).detach().to(F64)
    hidden = _norm(hidden, model.embedding_norm).detach()
    leaves = []
    for layer in model.layers:
        linears = [_Exact(m) for m in _projections(layer)]
        leaves += _leaves(*linears)
        hidden = _exact_bert(layer, hidden, linears)
    emb = F.normalize(hidden.mean(1), dim=-1)
    b = case["batch"]
    logits = step.scale * (emb[:b] @ emb[b:].t())
    loss = F.cross_entropy(logits, torch.arange(b, device=logits.device))
    grad = torch.cat([g.reshape(-1) for g in torch.autograd.grad(loss, leaves)])
    norm = grad.norm()
    return loss.detach(), norm, grad * torch.clamp(step.max_grad_norm / norm, max=1.0)
