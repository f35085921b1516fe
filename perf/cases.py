"""The work a program has this framework do, as cases that can be timed and checked.

Each case is one call (or the two or three calls of one block, or one pass of a
whole model) through the package's public entry points, over the sizes its
configurations, tests and benchmark use: W4A16 linears from one row to a prompt
batch of 8192, prompt attention of a fresh batch and of a later chunk of one long
prompt, decode attention of many and of one long sequence, a decode step of a model
replayed as a HIP graph, and a prompt pass of a model.

``exact`` computes the same in float64 with torch alone.
"""

from __future__ import annotations

import math

import torch

from torch2iron_amd import model as qwen
from torch2iron_amd import ops
from torch2iron_amd.formats import W4A16Weight

DEV = "cuda:0"
BF16 = torch.bfloat16
G = 128            # quantisation group
D = 128            # head dimension
EPS = 1e-6
THETA = 1e6

# hidden and intermediate sizes of the two decoders the package configures, and
# the fused projection widths that follow (16 q heads, 8 kv heads of 128)
DECODERS = {1024: 3072, 2048: 6144}
QKV = 4096
VOCAB = 151936

# Decoder layers of the model cases.  The layers of a decoder are alike; eight of them
# keep a state quick to make and the last layer's values near the float64 ones.
LAYERS = 8


def listed():
    return [
        # the smallest call: one token's output projection with its residual (single stream)
        {"name": "linear_1", "kind": "linear", "m": 1, "k": 2048, "n": 1024, "residual": True},
        # one short chat prompt: its fused q|k|v projection
        {"name": "linear_197_qkv", "kind": "linear", "m": 197, "k": 2048, "n": 4096, "residual": False},
        # the MLP block of a somewhat longer prompt
        {"name": "mlp_331", "kind": "mlp", "m": 331, "hidden": 2048},
        # a long prompt's down projection, ragged row count
        {"name": "linear_4001_down", "kind": "linear", "m": 4001, "k": 6144, "n": 2048, "residual": True},
        # the largest call: gate and up with SwiGLU over a prompt batch (16 x 512 tokens)
        {"name": "gate_up_8192", "kind": "gate_up", "m": 8192, "k": 2048, "inter": 6144},
        # the prompt batch's q|k|v projection with its q/k norm, RoPE and cache write
        {"name": "qkv_rope_16x512", "kind": "qkv_rope", "b": 16, "t": 512, "p0": 0, "hidden": 1024, "cap": 640},
        # the prompt batch's causal attention
        {"name": "prefill_attention_16x512", "kind": "prefill_attention", "b": 16, "t": 512, "p0": 0, "hq": 16,
         "hkv": 8, "cap": 640},
        # a later chunk of one long prompt, four q heads a kv head, odd length and start
        {"name": "prefill_attention_chunk", "kind": "prefill_attention", "b": 1, "t": 1999, "p0": 6001, "hq": 32,
         "hkv": 8, "cap": 8192},
        # a serving batch of sequences of differing lengths
        {"name": "decode_attention_32x4096", "kind": "decode_attention", "b": 32, "hq": 16, "hkv": 8, "cap": 4096,
         "lo": 1500, "hi": 4090},
        # one long document, one sequence
        {"name": "decode_attention_1x32768", "kind": "decode_attention", "b": 1, "hq": 32, "hkv": 8, "cap": 32768,
         "lo": 30011, "hi": 30011},
        # batched greedy decode: one step of a model with its head, replayed as a graph
        {"name": "decode_step_16", "kind": "decode_step", "b": 16, "cap": 640, "lo": 512, "hi": 600, "hidden": 1024},
        # one prompt pass of a model up to the first token's logits
        {"name": "prefill_model_3x211", "kind": "prefill_model", "b": 3, "t": 211, "hidden": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "gate_up", "qkv_rope", "prefill_attention",
                       "prefill_attention", "decode_attention", "decode_attention", "decode_step", "prefill_model"])
    hidden = rng.choice(sorted(DECODERS))
    if kind == "linear":
        k, n = rng.choice([(hidden, QKV), (2048, hidden), (DECODERS[hidden], hidden)])
        return {"kind": kind, "m": _log(rng, 1, 8192), "k": k, "n": n, "residual": n == hidden}
    if kind == "mlp":
        return {"kind": kind, "m": _log(rng, 1, 2048), "hidden": hidden}
    if kind == "gate_up":
        return {"kind": kind, "m": _log(rng, 1, 8192), "k": hidden, "inter": DECODERS[hidden]}
    if kind == "qkv_rope":
        b = rng.choice([1, 2, 3, 4, 8, 16])
        t = _log(rng, -(-512 // b), 8192 // b)
        p0 = rng.choice([0, 0, rng.randrange(1, 513)])
        return {"kind": kind, "b": b, "t": t, "p0": p0, "hidden": hidden, "cap": t + p0 + rng.randrange(0, 128)}
    if kind == "prefill_attention":
        b = rng.choice([1, 1, 2, 5, 16])
        hkv, q = rng.choice([(8, 2), (8, 4), (8, 1), (4, 8)])
        t = _log(rng, 17, 2048 if b < 5 else 512)
        p0 = rng.choice([0, rng.randrange(1, 6001 if b == 1 else 513)])
        return {"kind": kind, "b": b, "t": t, "p0": p0, "hq": hkv * q, "hkv": hkv, "cap": t + p0 + rng.randrange(0, 200)}
    if kind == "decode_attention":
        b = _log(rng, 1, 64)
        cap = _log(rng, 256, min(32768, 131072 // b))
        hkv, q = rng.choice([(8, 2), (8, 4), (8, 1), (4, 8)])
        hi = rng.randrange(cap // 2, cap)
        return {"kind": kind, "b": b, "hq": hkv * q, "hkv": hkv, "cap": cap, "lo": rng.randrange(cap // 4, hi), "hi": hi}
    if kind == "decode_step":
        cap = rng.choice([320, 640, 1088, 2048])
        hi = rng.randrange(cap // 2, cap)
        return {"kind": kind, "b": _log(rng, 1, 32), "cap": cap, "lo": rng.randrange(cap // 4, hi), "hi": hi,
                "hidden": hidden}
    b = rng.choice([1, 2, 3, 4, 8])
    return {"kind": kind, "b": b, "t": _log(rng, 16, 1536 // b), "hidden": hidden}


# ---- inputs, from the seed alone ----

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _words(nib):
    """Nibbles ``[..., 8]`` into int32 words, nibble j in bits 4 j .. 4 j + 3."""
    shifts = 4 * torch.arange(8, device=nib.device)
    w = (nib.to(torch.int64) << shifts).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)


def _quantised(g, k, n):
    """AutoGPTQ tensors of a linear with weights of standard deviation about 0.02:
    zero points near the middle of the range, values spread about them."""
    zero = torch.randint(6, 11, (k // G, n), device=DEV, generator=g)                     # effective zero point
    q = torch.randn(k // G, G, n, device=DEV, generator=g).mul_(2.7).add_(zero[:, None]).round_().clamp_(0, 15)
    qweight = _words(q.view(k // 8, 8, n).transpose(1, 2))
    qzeros = _words((zero - 1).view(k // G, n // 8, 8))
    scales = (torch.rand(k // G, n, device=DEV, generator=g) * 0.006 + 0.0045).to(torch.float16)
    return qweight.contiguous(), qzeros.contiguous(), scales


def _weight(parts):
    """A weight that stays resident: with its decode tiles, as the model loads it."""
    return ops.tile_weight(W4A16Weight(*parts))


def _pair(g, k, inter):
    """A gate|up weight: its columns alternate gate and up."""
    return _quantised(g, k, 2 * inter)


def _acts(g, *shape):
    """Activations: most channels near unit size, a few several times larger."""
    ch = torch.exp(0.5 * torch.randn(shape[-1], device=DEV, generator=g))
    return (torch.randn(*shape, device=DEV, generator=g) * ch).to(BF16)


def _norm_weight(g, n):
    return (0.9 + 0.2 * torch.rand(n, device=DEV, generator=g)).to(BF16)


def _rope(ctx):
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2).float() / D))
    ang = torch.outer(torch.arange(ctx).float(), inv)
    return torch.stack((torch.cos(ang), torch.sin(ang)), -1).reshape(ctx, D).to(BF16).to(DEV)


def _normal(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g).to(BF16)


def _positions(case):
    """The batch's positions, evenly from lo to hi (their order comes from the seed)."""
    b, lo, hi = case["b"], case["lo"], case["hi"]
    return [hi - (hi - lo) * i // max(b - 1, 1) for i in range(b)]


def _shuffled(g, case):
    pos = torch.tensor(_positions(case), dtype=torch.int32, device=DEV)
    return pos[torch.randperm(case["b"], device=DEV, generator=g)].contiguous()


def _inputs(case, seed):
    """Every tensor of a layer or block case."""
    g, kind = _gen(seed), case["kind"]
    s = {}
    if kind == "linear":
        s["w"] = _quantised(g, case["k"], case["n"])
        s["x"] = _acts(g, case["m"], case["k"])
        s["residual"] = _acts(g, case["m"], case["n"]) if case["residual"] else None
    elif kind == "gate_up":
        s["w"] = _pair(g, case["k"], case["inter"])
        s["x"] = _acts(g, case["m"], case["k"])
    elif kind == "mlp":
        h, inter = case["hidden"], DECODERS[case["hidden"]]
        s["w"], s["w_down"] = _pair(g, h, inter), _quantised(g, inter, h)
        s["norm"] = _norm_weight(g, h)
        s["x"] = _acts(g, case["m"], h)
    elif kind == "qkv_rope":
        s["w"] = _quantised(g, case["hidden"], QKV)
        s["x"] = _acts(g, case["b"] * case["t"], case["hidden"])
        s["q_norm"], s["k_norm"] = _norm_weight(g, D), _norm_weight(g, D)
        s["rope"] = _rope(case["cap"])
        s["k_cache"], s["v_cache"] = (_normal(g, case["b"], 8, case["cap"], D) for _ in range(2))
    elif kind == "prefill_attention":
        s["q"] = _normal(g, case["b"], case["hq"], case["t"], D)
        s["k_cache"], s["v_cache"] = (_normal(g, case["b"], case["hkv"], case["cap"], D) for _ in range(2))
    elif kind == "decode_attention":
        s["qkv"] = _acts(g, case["b"], (case["hq"] + 2 * case["hkv"]) * D)
        s["q_norm"], s["k_norm"] = _norm_weight(g, D), _norm_weight(g, D)
        s["rope"] = _rope(case["cap"])
        s["positions"] = _shuffled(g, case)
        s["k_cache"], s["v_cache"] = (_normal(g, case["b"], case["hkv"], case["cap"], D) for _ in range(2))
    return s


def _model_tensors(case, seed):
    """A decoder's tensors under their checkpoint names, on the GPU."""
    g, h = _gen(seed), case["hidden"]
    inter = DECODERS[h]
    t = {}

    def lin(name, k, n):
        t[f"{name}.qweight"], t[f"{name}.qzeros"], t[f"{name}.scales"] = _quantised(g, k, n)

    for i in range(LAYERS):
        p = f"model.layers.{i}"
        lin(f"{p}.self_attn.q_proj", h, 16 * D)
        lin(f"{p}.self_attn.k_proj", h, 8 * D)
        lin(f"{p}.self_attn.v_proj", h, 8 * D)
        lin(f"{p}.self_attn.o_proj", 16 * D, h)
        lin(f"{p}.mlp.gate_proj", h, inter)
        lin(f"{p}.mlp.up_proj", h, inter)
        lin(f"{p}.mlp.down_proj", inter, h)
        for nm, size in (("input_layernorm", h), ("post_attention_layernorm", h), ("self_attn.q_norm", D),
                         ("self_attn.k_norm", D)):
            t[f"{p}.{nm}.weight"] = _norm_weight(g, size)
    t["model.norm.weight"] = _norm_weight(g, h)
    t["model.embed_tokens.weight"] = _normal(g, VOCAB, h)
    return t


def _host(t):
    return {k: (v.float() if v.dtype == BF16 else v).cpu().numpy() for k, v in t.items()}


def _model_extra(case, seed):
    """Tokens, and for a decode step positions and the cache of the tokens before them."""
    g = _gen(seed + (1 << 32))
    if case["kind"] == "prefill_model":
        return {"prompt": torch.randint(0, VOCAB, (case["b"], case["t"]), device=DEV, generator=g, dtype=torch.int32)}
    shape = (LAYERS, case["b"], 8, case["cap"], D)
    return {"tokens": torch.randint(0, VOCAB, (case["b"],), device=DEV, generator=g, dtype=torch.int32),
            "positions": _shuffled(g, case), "k_cache": _normal(g, *shape), "v_cache": _normal(g, *shape)}


def _model_cap(case):
    return case["cap"] if case["kind"] == "decode_step" else case["t"] + 64


def prepare(case, seed):
    kind = case["kind"]
    if kind not in ("decode_step", "prefill_model"):
        s = _inputs(case, seed)
        for name in ("w", "w_down"):
            if name in s:
                s[name] = _weight(s[name])
        s["case"] = case
        if kind == "decode_attention":
            s["workspace"] = ops.Workspace()
        return s
    h = case["hidden"]
    cfg = qwen.Qwen3Config(hidden=h, intermediate=DECODERS[h], n_layers=LAYERS, vocab=VOCAB)
    m = qwen.Qwen3Model(_host(_model_tensors(case, seed)), cfg, batch=case["b"], ctx_cap=_model_cap(case), device=DEV)
    s = {"case": case, "model": m}
    extra = _model_extra(case, seed)
    if kind == "prefill_model":
        s["prompt"] = extra["prompt"]
        return s
    m.tokens.copy_(extra["tokens"])
    m.positions.copy_(extra["positions"])
    m.k_cache.copy_(extra["k_cache"])
    m.v_cache.copy_(extra["v_cache"])
    # a serving loop keeps its decode step as one graph; a step first outside the capture
    # makes the model's buffers
    m.forward_step(with_head=True, want_logits=True)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        m.forward_step(with_head=True, want_logits=True)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.linear(s["x"], s["w"], residual=s["residual"])
    if kind == "gate_up":
        return ops.gate_up(s["x"], s["w"])
    if kind == "mlp":
        if case["m"] <= 64:
            h = ops.rmsnorm_gate_up(s["x"], s["norm"], EPS, s["w"])
        else:
            h = ops.gate_up(ops.rmsnorm(s["x"], s["norm"], EPS), s["w"])
        return {"h": h, "y": ops.linear(h, s["w_down"], residual=s["x"])}
    if kind == "qkv_rope":
        q = ops.prefill_qkv_rope_kv(s["x"], s["w"], case["b"], case["p0"], 16, 8, s["q_norm"], s["k_norm"], EPS,
                                    s["rope"], s["k_cache"], s["v_cache"])
        return {"q": q, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "prefill_attention":
        return ops.prefill_attention(s["q"], case["p0"], case["hkv"], s["k_cache"], s["v_cache"])
    if kind == "decode_attention":
        ctx = ops.decode_attention(s["qkv"], s["positions"], case["hq"], case["hkv"], s["q_norm"], s["k_norm"], EPS,
                                   s["rope"], s["k_cache"], s["v_cache"], workspace=s["workspace"])
        return {"ctx": ctx, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    m = s["model"]
    if kind == "prefill_model":
        logits = m.prefill(s["prompt"], want_logits=True)
        return {"logits": logits, "k_cache": m.k_cache, "v_cache": m.v_cache}
    s["graph"].replay()
    return {"logits": m.logits, "x": m.x, "k_cache": m.k_cache, "v_cache": m.v_cache}


# ---- what a pass cannot do without ----

def _w_bytes(k, n):
    return k * n // 2 + (k // G) * n * 2 + (k // G) * n // 2


def _linear_work(m, k, n, out=None, residual=False):
    out = n if out is None else out
    return (_w_bytes(k, n) + 2 * m * (k + out + (out if residual else 0)), 2 * m * k * n)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        by, fl = _linear_work(case["m"], case["k"], case["n"], residual=case["residual"])
    elif kind == "gate_up":
        by, fl = _linear_work(case["m"], case["k"], 2 * case["inter"], out=case["inter"])
    elif kind == "mlp":
        m, h, inter = case["m"], case["hidden"], DECODERS[case["hidden"]]
        # x in, h and y out, both weights
        by = _w_bytes(h, 2 * inter) + _w_bytes(inter, h) + 2 * h + 2 * m * (2 * h + inter)
        fl = 2 * m * h * 3 * inter
    elif kind == "qkv_rope":
        m = case["b"] * case["t"]
        by, fl = _linear_work(m, case["hidden"], QKV)
        by += 2 * case["t"] * D
    elif kind == "prefill_attention":
        b, t, p0, hq, hkv = (case[k] for k in ("b", "t", "p0", "hq", "hkv"))
        by = 2 * D * b * (2 * hq * t + 2 * hkv * (p0 + t))
        fl = 4 * D * b * hq * (t * p0 + t * (t + 1) // 2)
    elif kind == "decode_attention":
        slots = sum(p + 1 for p in _positions(case))
        by = 2 * D * (2 * case["hkv"] * slots + case["b"] * (2 * case["hq"] + 2 * case["hkv"]))
        fl = 4 * D * case["hq"] * slots
    else:
        h, b = case["hidden"], case["b"]
        inter = DECODERS[h]
        rows = b * case.get("t", 1)
        if kind == "decode_step":
            kv = sum(p + 1 for p in _positions(case))
            pairs = kv
        else:
            kv = rows
            pairs = b * case["t"] * (case["t"] + 1) // 2
        weights = _w_bytes(h, QKV) + _w_bytes(2048, h) + _w_bytes(h, 2 * inter) + _w_bytes(inter, h)
        by = LAYERS * (weights + 2 * D * 2 * 8 * kv) + 2 * VOCAB * h + 4 * b * VOCAB + 2 * rows * h
        fl = LAYERS * (2 * rows * (h * QKV + 2048 * h + 3 * h * inter) + 4 * D * 16 * pairs) + 2 * b * VOCAB * h
    return {"bytes": by, "flops": fl}


# About four times the error against float64 that each path shows: bf16 outputs (1.7e-3 to
# 2.3e-3 for one product), two or three bf16 steps in a block, eight layers of them in a model.
TOLERANCE = {"linear": 1e-2, "gate_up": 1.5e-2, "mlp": 2.5e-2, "qkv_rope": 1.6e-2, "prefill_attention": 1e-2,
             "decode_attention": 1.7e-2, "decode_step": 4e-2, "prefill_model": 4e-2}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ---- the same in float64 ----

def _dense(parts):
    """``W^T [K, N]`` in float64 from the AutoGPTQ tensors."""
    qweight, qzeros, scales = parts
    shifts = 4 * torch.arange(8, device=qweight.device, dtype=torch.int32)
    k, n = qweight.shape[0] * 8, qweight.shape[1]
    q = ((qweight[:, None, :] >> shifts[:, None]) & 15).reshape(k // G, G, n)
    z = ((qzeros[:, :, None] >> shifts) & 15).reshape(k // G, 1, n) + 1
    return ((q - z).double() * scales.double()[:, None]).reshape(k, n)


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _silu_mul(gate, up):
    return gate * torch.sigmoid(gate) * up


def _paired(y):
    return _silu_mul(y[..., 0::2], y[..., 1::2])


def _rotate(x, ang):
    """RoPE over halves (i, i + D/2); ``ang`` ``[..., D]``, cos at even and sin at odd columns."""
    cos, sin = ang[..., 0::2].double(), ang[..., 1::2].double()
    a, b = x[..., : D // 2], x[..., D // 2:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _split_heads(y, b, t, hq, hkv):
    """A fused projection ``[b * t, (hq + 2 hkv) * D]`` into q, k, v ``[b, heads, t, D]``."""
    y = y.view(b, t, hq + 2 * hkv, D).transpose(1, 2)
    return y[:, :hq], y[:, hq:hq + hkv], y[:, hq + hkv:]


def _attend(q, k, v, mask):
    """Softmax attention ``q [b, hq, t, D]`` over ``k``, ``v [b, hkv, s, D]``; ``mask`` True where
    a key is seen, to broadcast over ``[b, 1, t, s]``.  One sequence and kv head at a time."""
    b, hq, t, _ = q.shape
    hkv = k.shape[1]
    out = torch.empty_like(q)
    for i in range(b):
        seen = mask[i if mask.shape[0] > 1 else 0, 0]
        for j in range(hkv):
            for r in range(hq // hkv):
                s = (q[i, j * (hq // hkv) + r] @ k[i, j].double().T) / math.sqrt(D)
                s.masked_fill_(~seen, -math.inf)
                out[i, j * (hq // hkv) + r] = torch.softmax(s, -1) @ v[i, j].double()
    return out


def _causal(t, p0, device):
    return (torch.arange(p0 + t, device=device)[None] <= torch.arange(p0, p0 + t, device=device)[:, None])[None, None]


def _decode_attend(y, s, hq, hkv, kc, vc, q_norm, k_norm):
    """One token a sequence: returns the context and the caches with the token's row."""
    b, cap = y.shape[0], kc.shape[2]
    pos = s["positions"].long()
    q, k, v = _split_heads(y, b, 1, hq, hkv)
    ang = s["rope"][pos][:, None, None]
    q, k = _rotate(_rms(q, q_norm), ang), _rotate(_rms(k, k_norm), ang)
    kc, vc = kc.double(), vc.double()
    rows = torch.arange(b, device=y.device)
    kc[rows, :, pos], vc[rows, :, pos] = k[:, :, 0], v[:, :, 0]
    mask = (torch.arange(cap, device=y.device)[None] <= pos[:, None])[:, None, None]
    return _attend(q, kc, vc, mask).transpose(1, 2).reshape(b, hq * D), kc, vc


def _exact_model(case, seed):
    t, s = _model_tensors(case, seed), _model_extra(case, seed)
    b, cap = case["b"], _model_cap(case)
    decode = case["kind"] == "decode_step"
    rows = 1 if decode else case["t"]
    ids = s["tokens"] if decode else s["prompt"].reshape(-1)
    emb = t["model.embed_tokens.weight"]
    x = emb[ids.long()].double()
    s["rope"] = _rope(cap)
    kcs, vcs = [], []

    def parts(name):
        return tuple(t[f"{name}.{f}"] for f in ("qweight", "qzeros", "scales"))

    for i in range(LAYERS):
        p = f"model.layers.{i}"
        xn = _rms(x, t[f"{p}.input_layernorm.weight"])
        y = torch.cat([xn @ _dense(parts(f"{p}.self_attn.{nm}_proj")) for nm in "qkv"], 1)
        qn, kn = t[f"{p}.self_attn.q_norm.weight"], t[f"{p}.self_attn.k_norm.weight"]
        if decode:
            ctx, kc, vc = _decode_attend(y, s, 16, 8, s["k_cache"][i], s["v_cache"][i], qn, kn)
        else:
            q, k, v = _split_heads(y, b, rows, 16, 8)
            ang = s["rope"][:rows]
            q, k = _rotate(_rms(q, qn), ang), _rotate(_rms(k, kn), ang)
            ctx = _attend(q, k, v, _causal(rows, 0, x.device)).transpose(1, 2).reshape(b * rows, 16 * D)
            kc, vc = (torch.nn.functional.pad(z, (0, 0, 0, cap - rows)) for z in (k, v))
        kcs.append(kc)
        vcs.append(vc)
        x = x + ctx @ _dense(parts(f"{p}.self_attn.o_proj"))
        xn = _rms(x, t[f"{p}.post_attention_layernorm.weight"])
        h = _silu_mul(xn @ _dense(parts(f"{p}.mlp.gate_proj")), xn @ _dense(parts(f"{p}.mlp.up_proj")))
        x = x + h @ _dense(parts(f"{p}.mlp.down_proj"))
    x = x.view(b, rows, -1)[:, -1]
    logits = _rms(x, t["model.norm.weight"]) @ emb.double().T
    out = {"logits": logits, "k_cache": torch.stack(kcs), "v_cache": torch.stack(vcs)}
    return dict(out, x=x) if decode else out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode_step", "prefill_model"):
        return _exact_model(case, seed)
    s = _inputs(case, seed)
    if kind == "linear":
        y = s["x"].double() @ _dense(s["w"])
        return y if s["residual"] is None else y + s["residual"].double()
    if kind == "gate_up":
        return _paired(s["x"].double() @ _dense(s["w"]))
    if kind == "mlp":
        x = s["x"].double()
        h = _paired(_rms(x, s["norm"]) @ _dense(s["w"]))
        return {"h": h, "y": h @ _dense(s["w_down"]) + x}
    if kind == "qkv_rope":
        b, t, p0 = case["b"], case["t"], case["p0"]
        q, k, v = _split_heads(s["x"].double() @ _dense(s["w"]), b, t, 16, 8)
        ang = s["rope"][p0:p0 + t]
        kc, vc = s["k_cache"].double(), s["v_cache"].double()
        kc[:, :, p0:p0 + t], vc[:, :, p0:p0 + t] = _rotate(_rms(k, s["k_norm"]), ang), v
        return {"q": _rotate(_rms(q, s["q_norm"]), ang), "k_cache": kc, "v_cache": vc}
    if kind == "prefill_attention":
        b, t, p0, hq = (case[k] for k in ("b", "t", "p0", "hq"))
        out = _attend(s["q"].double(), s["k_cache"][:, :, :p0 + t], s["v_cache"][:, :, :p0 + t], _causal(t, p0, DEV))
        return out.transpose(1, 2).reshape(b * t, hq * D)
    ctx, kc, vc = _decode_attend(s["qkv"].double(), s, case["hq"], case["hkv"], s["k_cache"], s["v_cache"],
                                 s["q_norm"], s["k_norm"])
    return {"ctx": ctx, "k_cache": kc, "v_cache": vc}
