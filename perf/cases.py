"""The work this library is measured on: single W4A16 projections, the quantizer, attention over a KV cache and the
fused decoder, each through the entry points a user's program calls, at sizes from the smallest call to a long prompt.

Every case is a dict of plain values with a "kind":

    linear     ops.linear(x [rows, k], W4Weight [n, k], bias)             layout "mma" (group 128 or 256) or "rows"
               (the canonical + v3 copies, any group of 32 j: what a weight whose K or group is no multiple of 128 uses)
    quantize   ops.quantize_w4_gpu(w [n, k], group, clip_grid)            a projection quantized at model load
    attention  ops.ext().attention(...)                                   `tokens` queries over `past` + `tokens` keys
    step       FusedDecoder.step: `tokens` tokens fed per graph replay after `past` cached ones
    prompt     FusedDecoder.prefill: a prompt of `tokens` tokens to its last position's logits

The decoders are slices of the Qwen2.5 architectures of lowbit.decode.QWEN25: all their widths and the whole head, a few
layers, random weights.
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.getcwd(), "lowbit-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from lowbit import decode, fused, ops  # noqa: E402

VOCAB = 151936
CLIP = (1.0, 0.975, 0.95, 0.925, 0.9, 0.875, 0.85, 0.825, 0.8, 0.775, 0.75)
HEADS = {"1.5b": (12, 2), "3b": (16, 2), "7b": (28, 4)}
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


def listed():
    return [
        # one eagerly launched decode token's attention-sized projection with its bias: launch and host latency
        {"name": "linear_1_row", "kind": "linear", "rows": 1, "k": 2048, "n": 2048, "group": 128, "layout": "mma",
         "bias": True},
        # a few requests decoded together through one MLP projection of the smallest benchmarked model
        {"name": "linear_13_rows", "kind": "linear", "rows": 13, "k": 1536, "n": 8960, "group": 128, "layout": "mma",
         "bias": False},
        # a larger decode batch (or a block of fed tokens) through a long-K projection
        {"name": "linear_48_rows", "kind": "linear", "rows": 48, "k": 11008, "n": 2048, "group": 128, "layout": "mma",
         "bias": False},
        # an ordinary prompt, ragged length, through a wide projection
        {"name": "linear_333_rows", "kind": "linear", "rows": 333, "k": 2048, "n": 11008, "group": 128, "layout": "mma",
         "bias": False},
        # a long prompt (or several batched) through the largest projection
        {"name": "linear_2048_rows", "kind": "linear", "rows": 2048, "k": 3584, "n": 18944, "group": 128,
         "layout": "mma", "bias": False},
        # a model quantized with groups of 64 (finer scales, the row-major kernels), a few rows
        {"name": "linear_group64", "kind": "linear", "rows": 6, "k": 896, "n": 4864, "group": 64, "layout": "rows",
         "bias": False},
        # loading a model: one projection quantized with the clip search
        {"name": "quantize_clip", "kind": "quantize", "n": 11008, "k": 2048, "group": 128, "dtype": "float16",
         "clip": True},
        # one decode token over a long context
        {"name": "attention_decode", "kind": "attention", "heads": "7b", "tokens": 1, "past": 16000},
        # a prompt's causal attention
        {"name": "attention_prompt", "kind": "attention", "heads": "3b", "tokens": 3000, "past": 0},
        # one greedy token of a decoder, replayed as a graph
        {"name": "step_1", "kind": "step", "model": "3b", "layers": 4, "tokens": 1, "past": 700},
        # sixteen tokens fed per step (scoring given text, verifying drafted tokens)
        {"name": "step_16", "kind": "step", "model": "3b", "layers": 4, "tokens": 16, "past": 512},
        # time to first token of a prompt
        {"name": "prompt_700", "kind": "prompt", "model": "3b", "layers": 4, "tokens": 700},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo .. hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["attention"] * 3 + ["quantize", "step", "prompt"])
    if kind == "linear":
        if rng.random() < 0.2:
            group = rng.choice([32, 64])
            k, n = group * _spread(rng, 8, 8192 // group), _spread(rng, 128, 8192)
            return {"kind": kind, "rows": _spread(rng, 1, 256), "k": k, "n": n, "group": group, "layout": "rows",
                    "bias": rng.random() < 0.5}
        k, n = 128 * _spread(rng, 4, 148), _spread(rng, 256, 22016)
        if rng.random() < 0.7:
            n = max(16, n // 16 * 16)
        rows = min(_spread(rng, 1, 2048), max(1, 2048 * 3584 * 18944 // (k * n)))
        return {"kind": kind, "rows": rows, "k": k, "n": n, "group": 128, "layout": "mma", "bias": rng.random() < 0.5}
    if kind == "quantize":
        group = rng.choice([32, 64, 128, 128, 128])
        return {"kind": kind, "n": _spread(rng, 128, 11008), "k": group * _spread(rng, 4, 4096 // group), "group": group,
                "dtype": rng.choice(sorted(DTYPES)), "clip": rng.random() < 0.6}
    if kind == "attention":
        heads = rng.choice(sorted(HEADS))
        tokens = _spread(rng, 1, 2048)
        past = _spread(rng, 1, max(1, min(16000, 2500 * 900 // tokens))) if rng.random() < 0.6 else 0
        return {"kind": kind, "heads": heads, "tokens": tokens, "past": past}
    model = rng.choice(["1.5b", "3b"])
    if kind == "step":
        return {"kind": kind, "model": model, "layers": rng.choice([2, 3, 4]), "tokens": rng.choice([1, 1, _spread(rng, 2, 64)]),
                "past": _spread(rng, 16, 1500)}
    return {"kind": kind, "model": model, "layers": rng.choice([2, 3, 4]), "tokens": _spread(rng, 8, 1000)}


# ---- inputs, from the seed alone ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 17)


def _normal(shape, gen, std=1.0, dtype=torch.float16):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dtype)


def _activations(rows, k, gen):
    """Unit-variance activations with a few large channels, as a transformer's residual stream has."""
    x = _normal((rows, k), gen, dtype=torch.float32)
    big = torch.rand(k, generator=gen, device="cuda") < 0.005
    return torch.where(big, 8.0 * x, x).half()


def _linear_inputs(case, seed):
    gen = _gen(seed)
    w = _normal((case["n"], case["k"]), gen, 0.02)
    x = _activations(case["rows"], case["k"], gen)
    return w, x, _normal((case["n"],), gen, 0.1) if case["bias"] else None


def _attention_inputs(case, seed):
    gen = _gen(seed)
    hq, hkv = HEADS[case["heads"]]
    t, keys = case["tokens"], case["past"] + case["tokens"]
    room = -(-keys // 64) * 64
    q = _normal((t, hq, 128), gen, 2.0)
    k, v = torch.zeros(2, hkv, room, 128, dtype=torch.float16, device="cuda")
    k[:, :keys] = _normal((hkv, keys, 128), gen)
    v[:, :keys] = _normal((hkv, keys, 128), gen)
    return q, k, v, torch.arange(case["past"], keys, device="cuda")


def _model(case, seed):
    """A decoder in the module layout of transformers' Qwen2ForCausalLM, which FusedQwen2 takes its weights from."""
    gen = _gen(seed)
    hidden, inter, _, hq, hkv = decode.QWEN25[case["model"]]

    def lin(n, k, bias=False):
        return SimpleNamespace(weight=_normal((n, k), gen, 0.02), bias=_normal((n,), gen, 0.1) if bias else None)

    def norm():
        return SimpleNamespace(weight=(1.0 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")).half())

    layers = []
    for _ in range(case["layers"]):
        att = SimpleNamespace(q_proj=lin(hq * 128, hidden, True), k_proj=lin(hkv * 128, hidden, True),
                              v_proj=lin(hkv * 128, hidden, True), o_proj=lin(hidden, hq * 128))
        mlp = SimpleNamespace(gate_proj=lin(inter, hidden), up_proj=lin(inter, hidden), down_proj=lin(hidden, inter))
        layers.append(SimpleNamespace(self_attn=att, mlp=mlp, input_layernorm=norm(), post_attention_layernorm=norm()))
    embed = SimpleNamespace(weight=_normal((VOCAB, hidden), gen, 0.02))
    inv_freq = 1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float32, device="cuda") / 128.0))
    config = SimpleNamespace(hidden_size=hidden, num_attention_heads=hq, num_key_value_heads=hkv, head_dim=128,
                             rms_norm_eps=1e-6)
    body = SimpleNamespace(embed_tokens=embed, norm=norm(), rotary_emb=SimpleNamespace(inv_freq=inv_freq), layers=layers)
    ids = torch.randint(0, VOCAB, (case.get("past", 0) + case["tokens"],), generator=gen, device="cuda")
    return SimpleNamespace(config=config, model=body, lm_head=embed), ids


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x, bias = _linear_inputs(case, seed)
        layouts = ("mma",) if case["layout"] == "mma" else ("canonical", "v3")
        return {"case": case, "x": x, "bias": bias, "w": ops.W4Weight.from_float(w, case["group"], layouts)}
    if kind == "quantize":
        w = _normal((case["n"], case["k"]), _gen(seed), 0.02, DTYPES[case["dtype"]])
        return {"case": case, "w": w}
    if kind == "attention":
        q, k, v, pos = _attention_inputs(case, seed)
        hq, hkv = HEADS[case["heads"]]
        out = torch.empty(case["tokens"], hq * 128, dtype=torch.float16, device="cuda")
        return {"case": case, "q": q, "k": k, "v": v, "pos": pos, "out": out, "hq": hq, "hkv": hkv}
    model, ids = _model(case, seed)
    past = case.get("past", 0)
    dec = fused.FusedDecoder(fused.FusedQwen2(model, past + case["tokens"] + 32), case["tokens"] if kind == "step" else 1)
    if kind == "step":
        dec.prefill(ids[:past])
        dec.capture()
    return {"case": case, "dec": dec, "ids": ids[past:].clone()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.linear(state["x"], state["w"], bias=state["bias"])
    if kind == "quantize":
        return ops.quantize_w4_gpu(state["w"], case["group"], CLIP if case["clip"] else None)
    if kind == "attention":
        ops.ext().attention(state["q"], state["k"], state["v"], state["pos"], state["out"], state["hq"], state["hkv"],
                            state["k"].shape[1], 128 ** -0.5)
        return state["out"]
    if kind == "step":
        state["dec"].pos = case["past"]          # every pass feeds the same tokens at the same positions
        return state["dec"].step(state["ids"])
    return state["dec"].prefill(state["ids"])


# ---- what a pass cannot do without ----

def _linear_work(rows, k, n, group, extra=0):
    return (n * k // 2 + 2 * n * (k // group) + 2 * rows * (k + n) + extra, 2 * rows * k * n)


def _attention_pairs(tokens, past):
    return tokens * past + tokens * (tokens + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "linear":
        b, f = _linear_work(case["rows"], case["k"], case["n"], case["group"], 2 * case["n"] if case["bias"] else 0)
    elif kind == "quantize":
        size = case["n"] * case["k"]
        b = size * (4 if case["dtype"] == "float32" else 2) + size // 2 + 2 * size // case["group"]
        f = size * (8 * len(CLIP) if case["clip"] else 4)
    elif kind == "attention":
        hq, hkv = HEADS[case["heads"]]
        b = 4 * case["tokens"] * hq * 128 + 4 * hkv * (case["past"] + case["tokens"]) * 128
        f = 4 * _attention_pairs(case["tokens"], case["past"]) * hq * 128
    else:
        hidden, inter, _, hq, hkv = decode.QWEN25[case["model"]]
        m, past = case["tokens"], case.get("past", 0)
        shapes = [(hidden, (hq + 2 * hkv) * 128), (hq * 128, hidden), (hidden, 2 * inter), (inter, hidden)]
        b = f = 0
        for k, n in shapes:
            b += n * k // 2 + 2 * n * (k // 128)
            f += 2 * m * k * n
        b += 4 * hkv * (past + m) * 128                 # the layer's cache
        f += 4 * _attention_pairs(m, past) * hq * 128
        head_rows = m if kind == "step" else 1
        b, f = case["layers"] * b, case["layers"] * f
        b += 2 * VOCAB * hidden + 2 * head_rows * VOCAB + 2 * m * hidden
        f += 2 * head_rows * VOCAB * hidden
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    # about four times the error against exact() below
    if kind == "linear":                                # fp16 outputs, weights rounded to fp16 or not: 2.1e-4 .. 3.4e-4
        return {"rel": 1.3e-3, "max": 6e-3}
    if kind == "attention":                             # fp16 outputs, fp32 softmax and sums: 2.1e-4
        return {"rel": 9e-4, "max": 6e-3}
    return {"rel": 8e-3, "max": 5e-2}                   # logits after layers of fp16 activations: 2.0e-3


# ---- the same in 64 bits ----

def _quantized(w, group, clip=None):
    """(q - 8 as float64 [n, k / group, group], scales float64 [n, k / group, 1], packed bytes, fp16 scales) by the
    format's rule: scale = fp16(fp32 amax / 7) (1 for an all-zero group), q = round_half_even(fp32 w / scale)."""
    n, k = w.shape
    wf = w.float().view(n, k // group, group)
    amax = wf.abs().amax(-1, keepdim=True)
    s = (amax / 7.0).half()
    s = torch.where(s == 0, torch.ones_like(s), s)
    q = torch.clamp(torch.round(wf / s.float()), -8, 7)
    u = (q + 8).to(torch.uint8).view(n, k // 2, 2)
    return q.double(), s.double(), u[..., 0] | (u[..., 1] << 4), s.view(n, k // group)


def _dequantized(w, group=128):
    q, s, _, _ = _quantized(w, group)
    return (q * s).view(w.shape)


def _attend(q, k, v, first):
    """Causal attention in float64: q [t, hq, 128] at positions first .., k and v [hkv, keys, 128]."""
    t, hq, _ = q.shape
    per = hq // k.shape[0]
    out = torch.empty(t, hq, 128, dtype=torch.float64, device=q.device)
    pos = torch.arange(first, first + t, device=q.device)
    mask = torch.arange(k.shape[1], device=q.device)[None, :] > pos[:, None]
    for h in range(hq):
        s = (q[:, h].double() @ k[h // per].double().t().contiguous()) * 128 ** -0.5
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ v[h // per].double()
    return out.reshape(t, hq * 128)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()


def _rope(x, inv_freq):
    """x [t, heads, 128] at positions 0 .. t - 1, the angles in fp32 and their cos and sin in fp16, as fp16 models do."""
    ang = torch.arange(x.shape[0], device=x.device, dtype=torch.float32)[:, None] * inv_freq[None, :]
    c, s = ang.cos().half().double()[:, None], ang.sin().half().double()[:, None]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _logits(case, seed, last):
    model, ids = _model(case, seed)
    body, cfg = model.model, model.config
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    h = body.embed_tokens.weight[ids].double()

    def lin(x, m):
        y = x @ _dequantized(m.weight).t()
        return y if m.bias is None else y + m.bias.double()

    for layer in body.layers:
        att, mlp = layer.self_attn, layer.mlp
        x = _rms(h, layer.input_layernorm.weight)
        q, k, v = (lin(x, m).view(x.shape[0], -1, 128) for m in (att.q_proj, att.k_proj, att.v_proj))
        q, k = _rope(q, body.rotary_emb.inv_freq), _rope(k, body.rotary_emb.inv_freq)
        h = h + lin(_attend(q, k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), 0), att.o_proj)
        x = _rms(h, layer.post_attention_layernorm.weight)
        h = h + lin(torch.nn.functional.silu(lin(x, mlp.gate_proj)) * lin(x, mlp.up_proj), mlp.down_proj)
    return _rms(h[-last:], body.norm.weight) @ model.lm_head.weight.double().t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x, bias = _linear_inputs(case, seed)
        y = x.double() @ _dequantized(w, case["group"]).t()
        return y if bias is None else y + bias.double()
    if kind == "quantize":
        if case["clip"]:
            return None                                 # the search's choice between near-equal errors is fp32's
        _, _, packed, scales = _quantized(_normal((case["n"], case["k"]), _gen(seed), 0.02, DTYPES[case["dtype"]]),
                                          case["group"])
        return packed, scales
    if kind == "attention":
        q, k, v, _ = _attention_inputs(case, seed)
        keys = case["past"] + case["tokens"]
        return _attend(q, k[:, :keys], v[:, :keys], case["past"])
    if kind == "step":
        return _logits(case, seed, case["tokens"])
    return _logits(case, seed, 1)[0]
