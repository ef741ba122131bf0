"""The work that callers of this framework have it do, as cases that can be timed and compared.

A case is one call (or one stack of calls) through the package's public entry points on layers of
the shapes in `hydra_amd.formats`:

  layer      one mixture-of-experts layer over T tokens (`MoELayer.forward_into`): T = 1 to 16 is
             decode of one stream or of a few streams together, larger T a prompt or one chunk
             of a long prompt;
  stack      the FFN blocks of consecutive layers on one fp32 residual stream
             (`Runner.forward`), as a model's forward pass runs them;
  attention  one token's attention over its key/value history (`attention_decode_into`).

`draw` takes the same kinds over T = 1..2048 and 128..131072 keys. Every state holds weights,
inputs and outputs of its own; all states share one context, as a program has one.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hydra_amd import formats as F
from hydra_amd.attention import attention_decode_into
from hydra_amd.layer import Context, MoELayer, Runner

MXFP4, MLX4, MLX8, BF16 = F.QUANT_MXFP4, F.QUANT_MLX4, F.QUANT_MLX8, F.QUANT_BF16
FAMILIES = ["gpt-oss-20b", "gpt-oss-120b", "qwen-35b-a3b-q4", "qwen-35b-a3b-q8", "gemma-bf16"]
ZIPF = 1.1          # skew of the expert load in chunked prefill of the 128-expert MXFP4 layer
Q_HEADS, KV_HEADS = 64, 8


def listed():
    return [
        # One token of one stream: the latency a reader of the generated text sees.
        {"name": "oss20_decode_1", "kind": "layer", "config": "gpt-oss-20b", "tokens": 1, "zipf": 0.0},
        # Eight streams decoded together.
        {"name": "oss20_decode_8", "kind": "layer", "config": "gpt-oss-20b", "tokens": 8, "zipf": 0.0},
        # A whole token through the MoE halves of the 24-layer model.
        {"name": "oss20_stack_24", "kind": "stack", "config": "gpt-oss-20b", "tokens": 1, "layers": 24},
        # A short prompt of ragged length: five or six tokens an expert.
        {"name": "oss20_prompt_45", "kind": "layer", "config": "gpt-oss-20b", "tokens": 45, "zipf": 0.0},
        # A chunk of a long prompt through the larger layer, with a skewed expert load.
        {"name": "oss120_prefill_512", "kind": "layer", "config": "gpt-oss-120b", "tokens": 512, "zipf": ZIPF},
        # The largest chunk.
        {"name": "oss120_prefill_2048", "kind": "layer", "config": "gpt-oss-120b", "tokens": 2048, "zipf": ZIPF},
        # One token through the layer of many small 4-bit experts with its shared expert.
        {"name": "qwen4_decode_1", "kind": "layer", "config": "qwen-35b-a3b-q4", "tokens": 1, "zipf": 0.0},
        # A chunk of a prompt through the same layer.
        {"name": "qwen4_prefill_1024", "kind": "layer", "config": "qwen-35b-a3b-q4", "tokens": 1024, "zipf": 0.0},
        # A prompt of odd length through the 8-bit layer: about ten tokens an expert.
        {"name": "qwen8_prompt_333", "kind": "layer", "config": "qwen-35b-a3b-q8", "tokens": 333, "zipf": 0.0},
        # Four streams decoded together on unquantised weights.
        {"name": "gemma_decode_4", "kind": "layer", "config": "gemma-bf16", "tokens": 4, "zipf": 0.0},
        # A long prompt's chunk on unquantised weights.
        {"name": "gemma_prefill_2048", "kind": "layer", "config": "gemma-bf16", "tokens": 2048, "zipf": 0.0},
        # One token's attention over a long history.
        {"name": "attention_32768", "kind": "attention", "keys": 32768, "head_dim": 64, "ring": 0, "start": 0},
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, its logarithm uniform."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["layer"] * 7 + ["stack"] + ["attention"] * 2)
    if kind == "attention":
        keys = _spread(rng, 128, 131072)
        # A sliding-window layer keeps its keys in a ring that the visible ones wrap round.
        ring = keys + rng.randrange(0, 64) if keys <= 4096 and rng.random() < 0.5 else 0
        return {"kind": kind, "keys": keys, "head_dim": rng.choice([64, 64, 128]), "ring": ring,
                "start": rng.randrange(0, 10000) if ring else 0}
    config = rng.choice(FAMILIES)
    if kind == "stack":
        return {"kind": kind, "config": config, "tokens": _spread(rng, 1, 64), "layers": rng.randrange(2, 5)}
    tokens = _spread(rng, 1, 2048)
    return {"kind": kind, "config": config, "tokens": tokens,
            "zipf": ZIPF if config == "gpt-oss-120b" and tokens > 16 else 0.0}


# ---- inputs ------------------------------------------------------------------------------------

def _generator(seed, part):
    return torch.Generator(device="cuda:0").manual_seed((int(seed) * 1000003 + part) & 0x7FFFFFFFFFFF)


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda:0").normal_(mean, std, generator=g)


def _bytes(g, shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda:0", generator=g)


def _affine(g, count, rows, cols, bits, scale_mean, scale_std):
    """`count` MLX-affine matrices: code words, group scales, group biases (64 columns a group)."""
    centre = 7.5 if bits == 4 else 127.5
    words = _bytes(g, (count, rows, cols * bits // 8))
    scales = _normal(g, (count, rows, cols // 64), scale_std, scale_mean).abs()
    return [words, scales, (scales.float() * -centre).bfloat16()]


def _experts(g, desc, count, inter, small=False):
    """The tensors of `count` experts in the order of a blob's slots. `small`: down weights that
    keep a block's output well below the residual, as a trained stack does."""
    H, quant = desc.hidden, desc.quant
    if quant == MXFP4:
        out = []
        for rows, cols, low in ((2 * inter, H, 119), (H, inter, 112 if small else 119)):
            out += [_bytes(g, (count, rows, cols // 32, 16)),
                    torch.randint(low, low + 5, (count, rows, cols // 32), dtype=torch.uint8, device="cuda:0", generator=g),
                    _normal(g, (count, rows), 0.02)]
        return out
    if quant == BF16:
        return [_normal(g, (count, 2 * inter, H), 0.02), _normal(g, (count, H, inter), 0.02)]
    bits = 4 if quant == MLX4 else 8
    scale = 0.01 if bits == 4 else 0.01 / 17      # the same spread of values from 256 codes
    return [t for rows, cols in ((inter, H), (inter, H), (H, inter))
            for t in _affine(g, count, rows, cols, bits, scale, 0.2 * scale)]


def _layer_tensors(desc, seed, part, zipf=0.0, small=False):
    """One layer's weights as separate tensors on the GPU."""
    g = _generator(seed, 100 + part)
    H, E = desc.hidden, desc.experts
    t = {"experts": _experts(g, desc, E, desc.intermediate, small)}
    if desc.shared_intermediate:
        # The published quantised builds store this router and gate as 8-bit affine rows.
        t["shared"] = _experts(g, desc, 1, desc.shared_intermediate)
        s = 1.0 / (math.sqrt(H) * 255 / math.sqrt(12.0))
        t["router"] = [x[0] for x in _affine(g, 1, E, H, 8, s, 0.2 * s)]
        t["gate"] = [x[0] for x in _affine(g, 1, 1, H, 8, s, 0.2 * s)]
    elif desc.router == F.ROUTER_GEMMA:
        t["router"] = _normal(g, (E, H))
        t["scale"] = _normal(g, (H,), 0.1, 1.0)
        t["expert_scale"] = _normal(g, (E,), 0.1, 1.0)
    else:
        t["router"] = _normal(g, (E, H), 1.0 / math.sqrt(H))
        if zipf:
            rank = torch.randperm(E, device="cuda:0", generator=g)
            t["bias"] = (-zipf * torch.log1p(rank.float())).bfloat16()
        else:
            t["bias"] = _normal(g, (E,), 0.02)
    return t


def _rmsnorm64(v, weight, eps):
    v = v.double()
    return v * (v.square().mean(-1, keepdim=True) + eps).rsqrt() * weight.double()


def _layer_inputs(desc, seed, tokens):
    """(x, router input or None): bf16 [T][H]. The scaled-norm router reads the residual, the
    experts its norm."""
    g = _generator(seed, 7)
    if desc.router != F.ROUTER_GEMMA:
        return _normal(g, (tokens, desc.hidden)), None
    residual = _normal(g, (tokens, desc.hidden), 3.0)
    return _rmsnorm64(residual, torch.ones(desc.hidden, device="cuda:0"), 1e-6).bfloat16(), residual


def _block_inputs(desc, seed, tokens, layers):
    """(residual fp32 [T][H], per layer its norms (and the dense branch's output))."""
    g = _generator(seed, 8)
    H = desc.hidden
    hidden = torch.randn((tokens, H), device="cuda:0", generator=g) * 3
    norms = []
    for _ in range(layers):
        n = {"pre_norm": _normal(g, (H,), 0.1, 1.0), "eps": 1e-6 if desc.router == F.ROUTER_GEMMA else 1e-5}
        dense = None
        if desc.router == F.ROUTER_GEMMA:
            for k in ("post_expert_norm", "post_dense_norm", "post_norm"):
                n[k] = _normal(g, (H,), 0.1, 1.0)
            n["layer_scalar"] = _normal(g, (1,), 0.05, 0.9)
            dense = torch.randn((tokens, H), device="cuda:0", generator=g)
        norms.append((n, dense))
    return hidden, norms


def _attention_inputs(case, seed):
    g = _generator(seed, 9)
    d, rows = case["head_dim"], case["ring"] or case["keys"]
    q = torch.randn((Q_HEADS, d), device="cuda:0", generator=g)
    k = torch.randn((rows, KV_HEADS, d), device="cuda:0", generator=g).half()
    v = torch.randn((rows, KV_HEADS, d), device="cuda:0", generator=g).half()
    return q, k, v, _normal(g, (Q_HEADS,))


# ---- states and passes ---------------------------------------------------------------------------

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def _bits(t):
    return t.view(torch.int16) if t is not None and t.dtype == torch.bfloat16 else t


def _blobs(desc, tensors, inter):
    lay = F.blob_layout(desc, inter)
    blobs = torch.zeros((tensors[0].shape[0], lay.stride), dtype=torch.uint8, device="cuda:0")
    for off, size, t in zip(lay.offsets, lay.sizes, tensors):
        blobs[:, off:off + size] = t.reshape(t.shape[0], -1).view(torch.uint8)
    return blobs


def _resident(desc, t):
    named = {}
    if desc.shared_intermediate:
        named["shared_expert"] = _blobs(desc, t["shared"], desc.shared_intermediate)[0]
        for name, (words, scales, biases) in (("router", t["router"]), ("shared_gate", t["gate"])):
            named[f"{name}_words"] = words.view(torch.int32)
            named[f"{name}_scales"], named[f"{name}_biases"] = _bits(scales), _bits(biases)
    else:
        named = {"router_weight": _bits(t["router"]), "router_bias": _bits(t.get("bias")),
                 "router_scale": _bits(t.get("scale")), "router_expert_scale": _bits(t.get("expert_scale"))}
    blobs = _blobs(desc, t["experts"], desc.intermediate)
    return MoELayer.resident(desc, blobs, blobs.shape[1], named, _ctx(),
                             router_bits=8 if desc.shared_intermediate else 0)


def prepare(case, seed):
    ctx = _ctx()
    if case["kind"] == "attention":
        q, k, v, sinks = _attention_inputs(case, seed)
        s = {"q": q, "k": k, "v": v, "sinks": _bits(sinks), "out": torch.empty_like(q), "case": case}
    elif case["kind"] == "layer":
        desc = F.CONFIGS[case["config"]]
        T = case["tokens"]
        x, xr = _layer_inputs(desc, seed, T)
        s = {"layer": _resident(desc, _layer_tensors(desc, seed, 0, case["zipf"])), "x": _bits(x), "xr": _bits(xr),
             "y": torch.empty((T, desc.hidden), dtype=torch.float32, device="cuda:0"),
             "idx": torch.empty((T, desc.top_k), dtype=torch.int32, device="cuda:0"),
             "w": torch.empty((T, desc.top_k), dtype=torch.float32, device="cuda:0")}
        ctx.reserve(desc, T)
    else:
        desc = F.CONFIGS[case["config"]]
        hidden, norms = _block_inputs(desc, seed, case["tokens"], case["layers"])
        layers = [(_resident(desc, _layer_tensors(desc, seed, i, small=True)),
                   {k: _bits(v) if torch.is_tensor(v) else v for k, v in n.items()}, dense)
                  for i, (n, dense) in enumerate(norms)]
        s = {"runner": Runner(ctx, layers), "embedded": hidden, "hidden": torch.empty_like(hidden)}
        s["runner"].reserve(case["tokens"])
    torch.cuda.synchronize()
    return s


def run(s):
    ctx = _ctx()
    if "layer" in s:
        s["layer"].forward_into(s["x"], s["y"], s["idx"], s["w"], x_router=s["xr"])
        return s["y"], s["idx"], s["w"]
    if "runner" in s:
        with torch.cuda.stream(ctx.stream):
            s["hidden"].copy_(s["embedded"])
        s["runner"].forward(s["hidden"])
        return s["hidden"]
    c = s["case"]
    return attention_decode_into(ctx, s["q"], s["k"], s["v"], s["sinks"], c["keys"], start_position=c["start"],
                                 ring_size=c["ring"], out=s["out"])


# ---- what a pass cannot do without ---------------------------------------------------------------

def _touched(desc, tokens, zipf):
    """Experts that a batch reaches, from logits of the inputs' distribution."""
    r = np.random.RandomState(3)
    logits = r.standard_normal((tokens, desc.experts))
    if zipf:
        logits -= zipf * np.log1p(np.arange(desc.experts))
    return np.unique(np.argpartition(-logits, desc.top_k - 1, axis=1)[:, :desc.top_k]).size


def _layer_work(desc, tokens, zipf):
    H, E, K = desc.hidden, desc.experts, desc.top_k
    nbytes = _touched(desc, tokens, zipf) * F.streamed_expert_bytes(desc)
    flops = 2.0 * tokens * (E * H + 3 * K * desc.intermediate * H)
    if desc.shared_intermediate:
        nbytes += F.streamed_expert_bytes(desc, desc.shared_intermediate) + (E + 1) * (H + H // 64 * 4)
        flops += 6.0 * tokens * desc.shared_intermediate * H
    else:
        nbytes += 2 * E * H
    return nbytes, flops


def work(case):
    if case["kind"] == "attention":
        n = case["keys"] * KV_HEADS * case["head_dim"]
        return {"bytes": 4 * n + 8 * Q_HEADS * case["head_dim"],
                "flops": 4.0 * case["keys"] * Q_HEADS * case["head_dim"]}
    desc = F.CONFIGS[case["config"]]
    T = case["tokens"]
    if case["kind"] == "layer":
        nbytes, flops = _layer_work(desc, T, case["zipf"])
        io = T * desc.hidden * (2 + 4) + T * desc.top_k * 8
        if desc.router == F.ROUTER_GEMMA:
            io += T * desc.hidden * 2
        return {"bytes": nbytes + io, "flops": flops}
    nbytes, flops = _layer_work(desc, T, 0.0)
    io = T * desc.hidden * 8
    if desc.router == F.ROUTER_GEMMA:
        nbytes += T * desc.hidden * 4
    return {"bytes": case["layers"] * nbytes + io, "flops": case["layers"] * flops}


def tolerance(case):
    # About four times the measured distance of the outputs from 64-bit results: 3.6e-5 for MXFP4
    # layers (activations as sums of fp8 terms), 4.9e-6 for MLX and 2.6e-6 for BF16 layers,
    # 4.1e-7 for attention.
    if case["kind"] == "attention":
        return {"rel": 2e-6, "max": 1e-4}
    if case["kind"] == "stack":
        # Each block rounds its input to bf16: a last bit in one layer flips roundings in the next
        # (2e-4 over 4 layers, 8e-4 over 24), and now and then a near tie of a router: then a
        # token goes to another expert, 1e-2 to 5e-2.
        return {"rel": 3e-2, "max": 0.99}
    rel = {MXFP4: 1.5e-4, BF16: 1e-5}.get(F.CONFIGS[case["config"]].quant, 2e-5)
    return {"rel": rel, "max": 40 * rel, "differ": 0.0}


# ---- the same in 64 bits -------------------------------------------------------------------------

_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _mxfp4_64(blocks, scales):
    table = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=blocks.device)
    b = blocks.long()
    v = table[torch.stack([b & 15, b >> 4], dim=-1)].flatten(-2)          # low nibble first
    return (v * torch.exp2(scales.double() - 127).unsqueeze(-1)).flatten(-2)


def _affine_64(words, scales, biases, bits):
    b = words.long()
    q = torch.stack([b & 15, b >> 4], dim=-1).flatten(-2) if bits == 4 else b
    q = q.double().unflatten(-1, (-1, 64))
    return (q * scales.double().unsqueeze(-1) + biases.double().unsqueeze(-1)).flatten(-2)


def _expert_64(desc, tensors, e, x):
    """One expert on the rows of x (64-bit)."""
    if desc.quant == MXFP4:
        up = x @ _mxfp4_64(tensors[0][e], tensors[1][e]).T + tensors[2][e].double()
        g, u = up[:, 0::2], up[:, 1::2]
        g, u = g.clamp(max=desc.swiglu_limit), u.clamp(-desc.swiglu_limit, desc.swiglu_limit)
        h = g * torch.sigmoid(desc.swiglu_alpha * g) * (u + 1)
        return h @ _mxfp4_64(tensors[3][e], tensors[4][e]).T + tensors[5][e].double()
    if desc.quant == BF16:
        up = x @ tensors[0][e].double().T
        g, u = up.chunk(2, dim=-1)
        h = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u
        return h @ tensors[1][e].double().T
    g, u, d = (_affine_64(*(t[e] for t in tensors[3 * m:3 * m + 3]), desc.bits) for m in range(3))
    g, u = x @ g.T, x @ u.T
    return (g * torch.sigmoid(g) * u) @ d.T


def _layer_64(desc, t, x, x_router):
    """(y, idx, w) of one layer for bf16 inputs."""
    x = x.double()
    xr = x if x_router is None else x_router.double()
    if desc.router == F.ROUTER_GEMMA:
        xr = xr * (xr.square().mean(-1, keepdim=True) + desc.router_eps).rsqrt()
        logits = (xr * t["scale"].double() * desc.hidden ** -0.5) @ t["router"].double().T
    elif desc.shared_intermediate:
        logits = xr @ _affine_64(*t["router"], 8).T
    else:
        logits = xr @ t["router"].double().T + t["bias"].double()
    top, idx = torch.sort(logits, dim=-1, descending=True, stable=True)
    top, idx = top[:, :desc.top_k], idx[:, :desc.top_k]
    w = torch.softmax(top, dim=-1)
    if desc.router == F.ROUTER_GEMMA:
        w = w * t["expert_scale"].double()[idx]
    y = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        rows, rank = torch.nonzero(idx == e, as_tuple=True)
        y.index_add_(0, rows, _expert_64(desc, t["experts"], e, x[rows]) * w[rows, rank].unsqueeze(1))
    if desc.shared_intermediate:
        gate = torch.sigmoid(x @ _affine_64(*t["gate"], 8).T)
        y += gate * _expert_64(desc, t["shared"], 0, x)
    return y, idx, w


def exact(case, seed):
    if case["kind"] == "attention":
        q, k, v, sinks = _attention_inputs(case, seed)
        pos = torch.arange(case["start"], case["start"] + case["keys"], device="cuda:0")
        if case["ring"]:
            pos = pos % case["ring"]
        out = []
        for h in range(KV_HEADS):
            group = Q_HEADS // KV_HEADS
            s = q[h * group:(h + 1) * group].double() @ k[pos, h].double().T / math.sqrt(case["head_dim"])
            s = torch.cat([s, sinks[h * group:(h + 1) * group].double().unsqueeze(1)], dim=1)
            out.append(torch.softmax(s, dim=1)[:, :-1] @ v[pos, h].double())
        return torch.cat(out)
    desc = F.CONFIGS[case["config"]]
    if case["kind"] == "layer":
        x, xr = _layer_inputs(desc, seed, case["tokens"])
        y, _, w = _layer_64(desc, _layer_tensors(desc, seed, 0, case["zipf"]), x, xr)
        return y, None, w
    hidden, norms = _block_inputs(desc, seed, case["tokens"], case["layers"])
    hidden = hidden.double()
    for i, (n, dense) in enumerate(norms):
        x = _rmsnorm64(hidden, n["pre_norm"], n["eps"]).bfloat16()
        gemma = desc.router == F.ROUTER_GEMMA
        y = _layer_64(desc, _layer_tensors(desc, seed, i, small=True), x, hidden.bfloat16() if gemma else None)[0]
        if gemma:
            both = _rmsnorm64(dense, n["post_dense_norm"], n["eps"]) + _rmsnorm64(y, n["post_expert_norm"], n["eps"])
            hidden = (hidden + _rmsnorm64(both, n["post_norm"], n["eps"])) * n["layer_scalar"].double()
        else:
            hidden = hidden + y
    return hidden
