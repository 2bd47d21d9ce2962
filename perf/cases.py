"""Performance cases of the framework: what a user's program calls, over the
sizes it calls them with.

Each case is a dict of plain values; ``prepare`` makes what the program
holds before the call (weights, plans, a model with its prompt), ``run`` is
one pass through the public entry points, and ``exact`` is the same result
in 64 bits from plain torch.  Shapes are the Qwen2.5-0.5B decoder's (hidden
896, intermediate 4864, 14 query and 2 KV heads of 64, vocabulary 151936)
and a wider one with 128-wide heads (hidden 1536, intermediate 8960, 12
query and 2 KV heads).
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "qwen2.5-jetson-inference_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import linear_hip  # noqa: E402
import model_hip  # noqa: E402
import synthetic  # noqa: E402

# hidden, intermediate, query heads, KV heads
SHAPES = {"896": (896, 4864, 14, 2), "1536": (1536, 8960, 12, 2)}
VOCAB = 151936


def listed():
    return [
        # The smallest call: one layer's seven independent W8A16 GEMVs, one
        # launch (a linear benchmark, or a caller that batches one layer).
        {"name": "gemv_plan_layer", "kind": "gemv_plan", "shape": "896", "layers": 1},
        # A token's Linear weights streamed once: 24 layers, 370 MB of int8.
        {"name": "gemv_plan_token", "kind": "gemv_plan", "shape": "896", "layers": 24},
        # The tied LM head of one token, logits and greedy token.
        {"name": "lm_head", "kind": "lm_head", "vocab": VOCAB, "k": 896},
        # A short prompt's Linears: a layer at 32 tokens.
        {"name": "gemm_plan_w8_32", "kind": "gemm_plan", "shape": "896", "m": 32, "w8": True},
        # An ordinary prompt of no round length, on BF16 weights.
        {"name": "gemm_plan_bf16_200", "kind": "gemm_plan", "shape": "896", "m": 200,
         "w8": False},
        # A long prompt's Linears: a layer at 512 tokens.
        {"name": "gemm_plan_w8_512", "kind": "gemm_plan", "shape": "896", "m": 512, "w8": True},
        # The reference's call pattern, one call per Linear, on a prompt near
        # 1024 tokens with BF16 weights (workspace for the long reduction).
        {"name": "gemm_calls_bf16_1001", "kind": "gemm_calls", "shape": "896", "m": 1001,
         "w8": False},
        # The MLP's first half on a prompt that nearly fills the default
        # context (2048), wider model.
        {"name": "gate_up_w8_2000", "kind": "gate_up", "shape": "1536", "m": 2000, "w8": True},
        # Causal attention of one layer: a 512-token prompt, 64-wide heads.
        {"name": "attention_512_64", "kind": "attention", "tokens": 512, "heads": 14,
         "kv_heads": 2, "head_dim": 64, "max_seq": 1024},
        # The same on a prompt that nearly fills the default context, 128-wide
        # heads.
        {"name": "attention_2000_128", "kind": "attention", "tokens": 2000, "heads": 12,
         "kv_heads": 2, "head_dim": 128, "max_seq": 2048},
        # Generation at the default context length: 16 tokens fed one by one
        # (as a sampling loop does), logits of the last.
        {"name": "decode_w8_1500", "kind": "decode", "shape": "896", "layers": 24,
         "vocab": VOCAB, "max_seq": 2048, "context": 1500, "steps": 16, "w8": True},
        # Time to first token of a 512-token prompt.
        {"name": "prefill_w8_512", "kind": "prefill", "shape": "896", "layers": 24,
         "vocab": VOCAB, "max_seq": 1024, "tokens": 512, "w8": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv_plan", "lm_head", "gemm_plan", "gemm_plan", "gemm_calls",
                       "gemm_calls", "gate_up", "attention", "attention", "decode", "prefill"])
    shape = rng.choice(["896", "1536"])
    w8 = rng.random() < 0.6
    if kind == "gemv_plan":
        return {"kind": kind, "shape": shape, "layers": _log(rng, 1, 24 if shape == "896" else 8)}
    if kind == "lm_head":
        return {"kind": kind, "vocab": _log(rng, 4000, VOCAB), "k": rng.choice([896, 1536])}
    if kind in ("gemm_plan", "gemm_calls", "gate_up"):
        return {"kind": kind, "shape": shape, "m": _log(rng, 2, 2000 if kind != "gate_up" else 1900),
                "w8": w8}
    if kind == "attention":
        tokens = _log(rng, 17, 1950)
        hd = rng.choice([64, 128])
        heads, kv = rng.choice([(14, 2), (16, 2), (8, 8), (16, 4)] if hd == 64
                               else [(12, 2), (8, 2), (8, 1)])
        return {"kind": kind, "tokens": tokens, "heads": heads, "kv_heads": kv, "head_dim": hd,
                "max_seq": rng.choice([tokens, max(tokens, 1024), max(tokens, 2048)])}
    layers = 24 if shape == "896" else 8
    max_seq = rng.choice([1024, 2048])
    if kind == "decode":
        return {"kind": kind, "shape": shape, "layers": layers, "vocab": VOCAB,
                "max_seq": max_seq, "context": _log(rng, 16, max_seq - 20),
                "steps": rng.randint(8, 14), "w8": w8}
    return {"kind": kind, "shape": shape, "layers": layers, "vocab": VOCAB, "max_seq": max_seq,
            "tokens": _log(rng, 8, max_seq - 8), "w8": w8}


# ------------------------------------------------------------- inputs --


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(g, shape, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(torch.bfloat16)


def _linear_shapes(shape):
    """(out, in) of one layer's Linears, by name."""
    h, inter, heads, kv = SHAPES[shape]
    kv_dim = kv * (h // heads)
    return {"q": (h, h), "k": (kv_dim, h), "v": (kv_dim, h), "o": (h, h), "gate": (inter, h),
            "up": (inter, h), "down": (h, inter)}


def _weight(g, n, k, w8):
    """One Linear: int8 with BF16 group-64 scales of N(0, 0.02), or BF16."""
    if not w8:
        return {"w": _normal(g, (n, k), 0.02), "s": None}
    q = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    s = (torch.randn((n, k // 64), generator=g, device="cuda").abs() * (0.02 / 127)).to(
        torch.bfloat16)
    return {"w": q, "s": s}


def _biased(name):
    return name in ("q", "k", "v")


def _model_tensors(case, seed):
    """A random-init model's tensors by archive name, on the GPU: weights
    N(0, 0.02), W8A16 as the exporter quantises them."""
    h, inter, heads, kv = SHAPES[case["shape"]]
    g = _gen(seed)
    t = {"model.embed_tokens.weight": _normal(g, (case["vocab"], h), 0.02),
         "model.norm.weight": _normal(g, (h,), 0.02) + 1}
    names = dict(zip(("q", "k", "v", "o", "gate", "up", "down"), synthetic.LINEARS))
    for layer in range(case["layers"]):
        p = "model.layers.%d." % layer
        t[p + "input_layernorm.weight"] = _normal(g, (h,), 0.02) + 1
        t[p + "post_attention_layernorm.weight"] = _normal(g, (h,), 0.02) + 1
        for short, (n, k) in _linear_shapes(case["shape"]).items():
            name = p + names[short] + ".weight"
            w = torch.randn((n, k), generator=g, device="cuda") * 0.02
            if case["w8"]:
                blocks = w.view(n, k // 64, 64)
                s = blocks.abs().amax(dim=2) / 127
                t[name] = (blocks / s[:, :, None]).round().clamp(-127, 127).to(
                    torch.int8).view(n, k)
                t[name + ".scale"] = s.to(torch.bfloat16)
            else:
                t[name] = w.to(torch.bfloat16)
            if _biased(short):
                t[p + names[short] + ".bias"] = _normal(g, (n,), 0.02)
    return t


def _config(case):
    h, inter, heads, kv = SHAPES[case["shape"]]
    return synthetic.ModelConfig(hidden_size=h, intermediate_size=inter,
                                 num_layers=case["layers"], num_heads=heads, num_kv_heads=kv,
                                 vocab_size=case["vocab"])


def _tokens(case, seed):
    """The prompt and, for a decode, the tokens fed after it."""
    count = case["tokens"] if case["kind"] == "prefill" else case["context"] + case["steps"]
    g = torch.Generator().manual_seed((int(seed) & 0x7FFFFFFF) + 1)
    return torch.randint(0, case["vocab"], (count,), generator=g).tolist()


def _inputs(case, seed):
    """The tensors of a case that is not a whole model."""
    kind, g = case["kind"], _gen(seed)
    if kind == "lm_head":
        return {"w": _normal(g, (case["vocab"], case["k"]), 0.02), "x": _normal(g, (case["k"],))}
    if kind == "attention":
        rows = (case["kv_heads"], case["max_seq"], case["head_dim"])
        return {"q": _normal(g, (case["tokens"], case["heads"], case["head_dim"])),
                "k": _normal(g, rows), "v": _normal(g, rows)}
    h, inter, _, _ = SHAPES[case["shape"]]
    if kind == "gate_up":
        return {"gate": _weight(g, inter, h, case["w8"]), "up": _weight(g, inter, h, case["w8"]),
                "x": _normal(g, (case["m"], h))}
    m, w8 = (1, True) if kind == "gemv_plan" else (case["m"], case["w8"])
    layers = []
    for _ in range(case.get("layers", 1)):
        layer = {}
        for name, (n, k) in _linear_shapes(case["shape"]).items():
            layer[name] = _weight(g, n, k, w8)
            layer[name]["b"] = _normal(g, (n,), 0.02) if _biased(name) else None
        layers.append(layer)
    # q, k, v read one input, o, gate and up, down one each (independent
    # GEMMs: a layer's inputs are given, not chained)
    x = {"h": _normal(g, (m, h)), "a": _normal(g, (m, h)), "n": _normal(g, (m, h)),
         "i": _normal(g, (m, inter))}
    return {"layers": layers, "x": x, "m": m}


_INPUT_OF = {"q": "h", "k": "h", "v": "h", "o": "a", "gate": "n", "up": "n", "down": "i"}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        model = model_hip.Qwen2Model(_config(case), _model_tensors(case, seed),
                                     "w8a16" if case["w8"] else "w16a16",
                                     max_sequence_length=case["max_seq"])
        state = {"kind": kind, "model": model, "tokens": _tokens(case, seed)}
        if kind == "decode":
            state["context"] = case["context"]
            model.prefill(state["tokens"][:case["context"]])
        return state
    state = _inputs(case, seed)
    state["kind"] = kind
    if kind == "lm_head":
        entries = linear_hip.lm_head_workspace_entries(case["vocab"], case["k"])
        state["logits"] = torch.empty(case["vocab"], dtype=torch.bfloat16, device="cuda")
        state["value"] = torch.empty(entries, dtype=torch.float32, device="cuda")
        state["index"] = torch.empty(entries, dtype=torch.int32, device="cuda")
        state["argmax"] = torch.empty(1, dtype=torch.int32, device="cuda")
        state["shape"] = (case["vocab"], case["k"])
    elif kind == "attention":
        state["out"] = torch.empty_like(state["q"])
        state["dims"] = (case["tokens"], case["heads"], case["kv_heads"], case["head_dim"],
                         case["max_seq"])
    elif kind == "gate_up":
        h, inter, _, _ = SHAPES[case["shape"]]
        state["out"] = torch.empty((case["m"], inter), dtype=torch.bfloat16, device="cuda")
        state["dims"] = (case["m"], inter, h)
        state["w8"] = case["w8"]
    else:
        m, calls = state["m"], []
        # a layer's outputs, one Linear's [m, n] after the other
        state["y"] = [torch.empty(m * sum(lin["w"].shape[0] for lin in layer.values()),
                                  dtype=torch.bfloat16, device="cuda")
                      for layer in state["layers"]]
        for layer, flat in zip(state["layers"], state["y"]):
            at = 0
            for name, lin in layer.items():
                n, k = lin["w"].shape
                x, y = state["x"][_INPUT_OF[name]], flat[at:at + m * n]
                at += m * n
                if kind == "gemv_plan":
                    calls.append((lin["w"], lin["s"], 64, lin["b"], x, y, n, k))
                elif case["w8"]:
                    calls.append((lin["w"], lin["s"], 64, lin["b"], x, y, m, n, k))
                else:
                    calls.append((lin["w"], lin["b"], x, y, m, n, k))
        if kind == "gemv_plan":
            state["plan"] = linear_hip.W8A16GemvPlan(calls)
        elif kind == "gemm_plan":
            state["plan"] = linear_hip.GemmPlan(calls)
        else:
            # one workspace for every Linear, sized for this many tokens
            need = max(linear_hip.gemm_workspace_bytes(m, c[-2], c[-1]) for c in calls)
            state["ws"] = torch.zeros(max(need, 256), dtype=torch.uint8, device="cuda")
            state["calls"] = calls
            state["call"] = linear_hip.gemm_w8a16_ws if case["w8"] else linear_hip.gemm_bf16_ws
    return state


# ---------------------------------------------------------------- run --


def run(state):
    kind = state["kind"]
    if kind == "prefill":
        model = state["model"]
        model.reset()
        model.prefill(state["tokens"])
        return model.last_logits_host()
    if kind == "decode":
        model, context, tokens = state["model"], state["context"], state["tokens"]
        model.rewind(context, tokens[context])
        for token in tokens[context:]:
            model.decode_next(token)
        return model.last_logits_host()
    if kind == "lm_head":
        vocab, k = state["shape"]
        linear_hip.lm_head_bf16(state["w"], None, state["x"], state["logits"], state["value"],
                                state["index"], state["argmax"], vocab, k)
        return {"logits": state["logits"], "argmax": state["argmax"]}
    if kind == "attention":
        model_hip.attention_prefill_bf16(state["q"], state["k"], state["v"], state["out"],
                                         *state["dims"])
        return state["out"]
    if kind == "gate_up":
        gate, up = state["gate"], state["up"]
        if state["w8"]:
            model_hip.gemm_gate_up_silu_w8a16(gate["w"], gate["s"], None, up["w"], up["s"], None,
                                              64, state["x"], state["out"], *state["dims"])
        else:
            model_hip.gemm_gate_up_silu_bf16(gate["w"], None, up["w"], None, state["x"],
                                             state["out"], *state["dims"])
        return state["out"]
    if kind == "gemm_calls":
        call, ws = state["call"], state["ws"]
        for c in state["calls"]:
            call(*c, ws)
    else:
        state["plan"].launch()
    return state["y"]


# --------------------------------------------------------------- work --


def work(case):
    """Each input read once, each output written once; multiply-adds as two."""
    kind = case["kind"]
    if kind == "lm_head":
        v, k = case["vocab"], case["k"]
        return {"bytes": 2.0 * v * k + 2 * k + 2 * v + 4, "flops": 2.0 * v * k}
    if kind == "attention":
        t, h, kv, d = case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
        return {"bytes": 2.0 * (2 * t * h * d + 2 * kv * t * d),
                "flops": 4.0 * h * d * t * (t + 1) / 2}
    h, inter, heads, kv = SHAPES[case["shape"]]
    w8 = case.get("w8", True)
    per = lambda n, k: n * k * (1 + 2 / 64) if w8 else 2.0 * n * k  # noqa: E731
    shapes = _linear_shapes(case["shape"])
    if kind == "gate_up":
        m = case["m"]
        return {"bytes": 2 * per(inter, h) + 2.0 * m * (h + inter), "flops": 4.0 * m * inter * h}
    weights = sum(per(n, k) for n, k in shapes.values())
    muls = sum(n * k for n, k in shapes.values())
    if kind in ("gemv_plan", "gemm_plan", "gemm_calls"):
        m, layers = case.get("m", 1), case.get("layers", 1)
        outs = sum(n for n, _ in shapes.values())
        return {"bytes": layers * (weights + 2.0 * m * outs) + 2.0 * m * (3 * h + inter),
                "flops": 2.0 * layers * m * muls}
    layers, vocab, kv_dim = case["layers"], case["vocab"], kv * (h // heads)
    if kind == "prefill":
        t = case["tokens"]
        return {"bytes": layers * (weights + 4.0 * t * kv_dim) + 2.0 * vocab * h + 2.0 * t * h,
                "flops": layers * (2.0 * t * muls + 4.0 * h * t * (t + 1) / 2) + 2.0 * vocab * h}
    steps, ctx = case["steps"], case["context"]
    return {"bytes": steps * (layers * (weights + 4.0 * (ctx + steps / 2) * kv_dim)
                              + 2.0 * vocab * h),
            "flops": steps * (layers * (2.0 * muls + 4.0 * h * (ctx + steps / 2)) + 2.0 * vocab * h)}


def tolerance(case):
    """BF16 outputs of FP32 sums: an output is off its exact value by up to
    half a BF16 unit (2^-9), about 1.7e-3 in the 2-norm; the whole models
    carry that through every layer."""
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 0.03, "max": 0.2}
    return {"rel": 7e-3, "max": 0.03, "differ": 0.0}


# -------------------------------------------------------------- exact --


def _f64(lin):
    w = lin["w"].double()
    if lin["s"] is None:
        return w
    n, k = w.shape
    return (w.view(n, k // 64, 64) * lin["s"].double()[:, :, None]).view(n, k)


def _attend(q, k, v):
    """Causal attention of q [t, heads, d] over k, v [kv, t, d], in 64 bits."""
    t, heads, d = q.shape
    mask = torch.ones((t, t), dtype=torch.bool, device=q.device).triu(1)
    out = torch.empty((t, heads, d), dtype=torch.float64, device=q.device)
    for h in range(heads):
        g = h // (heads // k.shape[0])
        s = (q[:, h] @ k[g].t().contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), dim=1) @ v[g]
    return out


def _exact_model(case, seed):
    """Logits of the last token, the whole sequence at once."""
    h, inter, heads, kv = SHAPES[case["shape"]]
    d, t = h // heads, _model_tensors(case, seed)
    tokens = torch.tensor(_tokens(case, seed), device="cuda")
    count = tokens.numel()

    def norm(x, w):
        return x / (x.square().mean(dim=1, keepdim=True) + 1e-6).sqrt() * w.double()

    def linear(x, name):
        y = x @ _f64({"w": t[name + ".weight"], "s": t.get(name + ".weight.scale")}).t()
        return y + t[name + ".bias"].double() if name + ".bias" in t else y

    pos = torch.arange(count, device="cuda", dtype=torch.float64)
    freq = 1e6 ** (-2.0 * torch.arange(d // 2, device="cuda", dtype=torch.float64) / d)
    cos, sin = (pos[:, None] * freq).cos()[:, None], (pos[:, None] * freq).sin()[:, None]

    def rope(x):
        a, b = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    x = t["model.embed_tokens.weight"][tokens].double()
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        n = norm(x, t[p + "input_layernorm.weight"])
        q = rope(linear(n, p + "self_attn.q_proj").view(count, heads, d))
        k = rope(linear(n, p + "self_attn.k_proj").view(count, kv, d))
        v = linear(n, p + "self_attn.v_proj").view(count, kv, d)
        a = _attend(q, k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous())
        x = x + linear(a.reshape(count, h), p + "self_attn.o_proj")
        n = norm(x, t[p + "post_attention_layernorm.weight"])
        m = torch.nn.functional.silu(linear(n, p + "mlp.gate_proj")) * linear(n, p + "mlp.up_proj")
        x = x + linear(m, p + "mlp.down_proj")
    last = norm(x[-1:], t["model.norm.weight"])[0]
    return (t["model.embed_tokens.weight"].double() @ last).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_model(case, seed)
    s = _inputs(case, seed)
    if kind == "lm_head":
        logits = s["w"].double() @ s["x"].double()
        return {"logits": logits, "argmax": logits.argmax().to(torch.int32).view(1)}
    if kind == "attention":
        t = case["tokens"]
        return _attend(s["q"].double(), s["k"][:, :t].double(), s["v"][:, :t].double())
    if kind == "gate_up":
        x = s["x"].double()
        return torch.nn.functional.silu(x @ _f64(s["gate"]).t()) * (x @ _f64(s["up"]).t())
    ys = []
    for layer in s["layers"]:
        outs = []
        for name, lin in layer.items():
            y = s["x"][_INPUT_OF[name]].double() @ _f64(lin).t()
            outs.append((y if lin["b"] is None else y + lin["b"].double()).view(-1))
        ys.append(torch.cat(outs))
    return ys
