"""The calls whose speed is tracked: DeepSeek-V2-Lite's decode and prompt path
through the public Python entry points of `fleet_moe`, on one GPU.

`listed()` holds the sizes this repository's tests and benchmark use, odd ones
beside them; `draw(rng)` gives more cases of the same ranges. Weights are
N(0, 0.02^2) bf16 in the packed layout, RMSNorm weights lie around 1, hidden
states are RMS-normed N(0, 1) vectors, all from the seed. `exact` evaluates a
case in 64 bits with plain torch, at the rounding points that define the
model's arithmetic (bf16 after every projection, RMSNorm and residual add).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent
if str(_ROOT / "fleet-mi300x_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "fleet-mi300x_amd"))

from fleet_moe import layout as _layout  # noqa: E402
from fleet_moe import ops  # noqa: E402
from fleet_moe import rope as _rope  # noqa: E402
from fleet_moe.layout import DSV2_LITE as _D  # noqa: E402

_DEV = "cuda"
_STD = 0.02
_H, _I, _SI, _E, _K = _D.hidden, _D.moe_inter, _D.shared_inter, _D.n_routed, _D.top_k
_HEADS, _LORA, _NOPE, _ROPE, _V = 16, 512, 128, 64, 128
_QKV = _HEADS * (_NOPE + _ROPE) + _LORA + _ROPE
_ROW = _LORA + _ROPE
_VOCAB, _DENSE, _LAYERS, _MAX_POS = _layout.VOCAB, _layout.DENSE_INTER, 27, 4096


def listed():
    return [
        # the router of one decoded token: the smallest call, all latency
        {"name": "route_1", "kind": "route", "tokens": 1},
        # the router of one prompt chunk or a large decode batch
        {"name": "route_250", "kind": "route", "tokens": 250},
        # one MoE layer of batch-1 decode, the path this library is built around
        {"name": "layer_1", "kind": "layer", "tokens": 1},
        # the attention half of a layer in batch-1 decode after a 1024-token prompt
        {"name": "attn_1024", "kind": "attn", "pos": 1024},
        # the same near the end of the KV cache, an odd position
        {"name": "attn_3967", "kind": "attn", "pos": 3967},
        # the dense layer 0 of batch-1 decode
        {"name": "dense_1", "kind": "dense", "tokens": 1},
        # lm_head and argmax of one decoded token, logits kept
        {"name": "lm_head_1", "kind": "lm_head", "tokens": 1},
        # router and experts of a small, ragged decode batch
        {"name": "moe_7", "kind": "moe", "tokens": 7},
        # the grouped experts of the benchmark's largest batch, skewed routing
        {"name": "grouped_64", "kind": "grouped", "tokens": 64},
        # router and experts of the largest batch one call takes
        {"name": "moe_256", "kind": "moe", "tokens": 256},
        # a whole decode step of the 27-layer model: one token's logits
        {"name": "step_1024", "kind": "step", "pos": 1024},
        # a prompt through the 27-layer model, and the first step after it
        {"name": "prompt_384", "kind": "prompt", "tokens": 384},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["route", "grouped", "moe", "attn", "step", "prompt"])
    if kind == "attn":
        return {"kind": kind, "pos": _log_int(rng, 1, _MAX_POS - 1)}
    if kind == "step":
        return {"kind": kind, "pos": _log_int(rng, 1, _MAX_POS - 1)}
    if kind == "prompt":
        return {"kind": kind, "tokens": _log_int(rng, 2, 384)}
    if kind == "route":
        return {"kind": kind, "tokens": _log_int(rng, 2, 512)}
    return {"kind": kind, "tokens": _log_int(rng, 1, 256)}


# ---------------------------------------------------------------- inputs

def _gen(seed, stream):
    g = torch.Generator(device=_DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) & (2**62 - 1))
    return g


def _fill(lay, seed):
    """Every tensor of `lay` in one packed device blob."""
    blob = torch.empty(lay.nbytes, dtype=torch.uint8, device=_DEV)
    g = _gen(seed, 1)
    w = blob.view(torch.bfloat16)
    step = 1 << 30
    for a in range(0, w.numel(), step):
        w[a: a + step].normal_(0.0, _STD, generator=g)
    for name, t in lay.tensors.items():
        if "norm" in name:
            v = w[t.offset // 2: (t.offset + t.nbytes) // 2]
            v.mul_(5.0).add_(1.0)                      # RMSNorm weights: 1 +- 0.1
    return blob


def _tensor(blob, lay, name):
    t = lay.tensors[name]
    return blob.view(torch.bfloat16)[t.offset // 2: (t.offset + t.nbytes) // 2]


def _vocab_layout(lay=None):
    lay = lay or _layout.Layout()
    lay.add("final_norm", (_H,))
    lay.add("lm_head", (_VOCAB, _H))
    return lay


def _attn_layout():
    lay = _layout.Layout()
    lay.add("L0.norm_in", (_H,))
    lay.add("L0.qkv", (_QKV, _H))
    lay.add("L0.kv_a_norm", (_LORA,))
    lay.add("L0.kv_b", (_HEADS * (_NOPE + _V), _LORA))
    lay.add("L0.o_proj", (_H, _HEADS * _V))
    return lay


def _dense_layout():
    lay = _layout.Layout()
    lay.add("L0.norm_post", (_H,))
    lay.add("L0.dense", (3 * _DENSE * _H,))
    return lay


def _normed(seed, tokens):
    """bf16-valued RMS-normed hidden states [tokens][H] in fp32."""
    x = torch.randn((tokens, _H), generator=_gen(seed, 2), device=_DEV)
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    return x.bfloat16().float()


def _residual(seed):
    """One token's residual stream, bf16-valued fp32 [H]."""
    return torch.randn(_H, generator=_gen(seed, 3), device=_DEV).bfloat16().float()


def _zipf_bias(seed):
    """A Zipf(1.1) prior over the experts, added to the router's logits."""
    perm = torch.randperm(_E, generator=_gen(seed, 4), device=_DEV)
    p = (torch.arange(_E, device=_DEV) + 1.0).pow(-1.1)
    return (p / p.sum()).log()[perm.argsort()].float()


def _cache_rows(seed, shape):
    return (0.5 * torch.randn(shape, generator=_gen(seed, 5), device=_DEV)).bfloat16()


def _tables():
    cos, sin = _rope.yarn_tables(_MAX_POS)
    return torch.from_numpy(cos).to(_DEV), torch.from_numpy(sin).to(_DEV)


def _inputs(case, seed):
    """The plain tensors of a case: packed weights and activations."""
    kind, s = case["kind"], {}
    if kind in ("route", "grouped", "moe", "layer"):
        s["lay"] = _layout.moe_layout(_D, layers=(1,))
        s["blob"] = _fill(s["lay"], seed)
        if kind == "layer":
            s["x"] = _residual(seed)
            return s
        s["x"] = _normed(seed, case["tokens"])
        if kind == "grouped":
            _, s["ids"], s["w"] = _route(_tensor(s["blob"], s["lay"], "L1.router"), s["x"],
                                         torch.float64, _zipf_bias(seed))
    elif kind == "attn":
        s["lay"] = _attn_layout()
        s["blob"] = _fill(s["lay"], seed)
        s["x"] = _residual(seed)
        s["cache"] = _cache_rows(seed, (_MAX_POS, _ROW))
    elif kind == "dense":
        s["lay"] = _dense_layout()
        s["blob"] = _fill(s["lay"], seed)
        s["x"] = _residual(seed)
    elif kind == "lm_head":
        s["lay"] = _vocab_layout()
        s["blob"] = _fill(s["lay"], seed)
        s["x"] = _residual(seed)
    else:
        s["lay"] = _layout.model_layout(_D, n_layers=_LAYERS)
        s["blob"] = _fill(s["lay"], seed)
        if kind == "step":
            s["rows"] = _cache_rows(seed, (_LAYERS, case["pos"], _ROW))
            n = 1
        else:
            n = case["tokens"]
        s["tokens"] = torch.randint(0, _VOCAB, (n,), generator=_gen(seed, 6), device=_DEV,
                                    dtype=torch.int32)
    return s


# ---------------------------------------------------------------- prepare, run

def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    s["kind"] = kind
    lay, blob = s["lay"], s["blob"]
    if kind in ("route", "grouped", "moe", "layer"):
        s["layer"] = ops.DeviceLayer(blob, lay, 1, _D)
        if kind == "layer":
            s["dec"] = ops.LayerDecoder(_D, device=_DEV)
            s["out"] = {"x_out": torch.empty(_H, device=_DEV),
                        "moe_out": torch.empty(_H, dtype=torch.int16, device=_DEV),
                        "ids": torch.empty(_K, dtype=torch.int32, device=_DEV),
                        "weights": torch.empty(_K, device=_DEV)}
        if kind in ("grouped", "moe"):
            s["runner"] = ops.GroupedRunner(case["tokens"], _D, device=_DEV)
        if kind == "grouped":
            s["x16"] = s["x"].bfloat16().view(torch.int16)
            s["ids"] = s["ids"].to(torch.int32)
            s["w"] = s["w"].float()
    elif kind == "attn":
        s["dec"] = ops.AttnDecoder(_D, device=_DEV)
        a = {n: blob.data_ptr() + t.offset for n, t in lay.tensors.items()}
        s["layer"] = ops._lib.FleetAttnLayer(a["L0.norm_in"], a["L0.qkv"], a["L0.kv_a_norm"],
                                             a["L0.kv_b"], a["L0.o_proj"])
        s["cos"], s["sin"] = _tables()
        s["cache16"] = s["cache"].view(torch.int16)
        s["x_out"] = torch.empty_like(s["x"])
        s["pos"] = case["pos"]
    elif kind == "dense":
        s["dec"] = ops.DenseDecoder(_D, _DENSE, device=_DEV)
        s["norm_ptr"] = blob.data_ptr() + lay.tensors["L0.norm_post"].offset
        s["dense_ptr"] = blob.data_ptr() + lay.tensors["L0.dense"].offset
        s["x_out"] = torch.empty_like(s["x"])
        s["mlp_out"] = torch.empty(_H, dtype=torch.int16, device=_DEV)
    elif kind == "lm_head":
        s["dec"] = ops.AttnDecoder(_D, device=_DEV)
        s["norm_ptr"] = blob.data_ptr() + lay.tensors["final_norm"].offset
        s["head_ptr"] = blob.data_ptr() + lay.tensors["lm_head"].offset
        s["logits"] = torch.empty(_VOCAB, device=_DEV)
        s["token"] = torch.empty(1, dtype=torch.int32, device=_DEV)
    else:
        s["dec"] = ops.Decoder(blob, lay, _D, max_pos=_MAX_POS)
        s["logits"] = torch.empty(_VOCAB, device=_DEV)
        if kind == "step":
            s["pos"] = case["pos"]
            s["dec"].cache[:, : case["pos"]] = s.pop("rows").view(torch.int16)
    return s


def run(s):
    kind = s["kind"]
    if kind == "route":
        return ops.route(s["layer"], s["x"])
    if kind == "layer":
        o = s["out"]
        s["dec"].decode_into(s["layer"], s["x"], o["x_out"], o["moe_out"], o["ids"], o["weights"])
        return {"x_out": o["x_out"], "moe_out": o["moe_out"].view(torch.bfloat16),
                "ids": o["ids"], "weights": o["weights"]}
    if kind == "grouped":
        return s["runner"].run(s["layer"], s["x16"], s["ids"], s["w"]).view(torch.bfloat16)
    if kind == "moe":
        r = ops.moe(s["layer"], s["x"], s["runner"])
        return {**r, "out": r["out"].view(torch.bfloat16)}
    if kind == "attn":
        s["dec"].attn_into(s["layer"], s["x"], s["x_out"], s["cache16"], s["pos"], None,
                           s["cos"], s["sin"])
        return {"x_out": s["x_out"], "row": s["cache"][s["pos"]]}
    if kind == "dense":
        s["dec"].decode_into(s["norm_ptr"], s["dense_ptr"], s["x"], s["x_out"], s["mlp_out"])
        return {"x_out": s["x_out"], "mlp_out": s["mlp_out"].view(torch.bfloat16)}
    if kind == "lm_head":
        s["dec"].lm_head_into(s["x"], s["norm_ptr"], s["head_ptr"], s["logits"], s["token"])
        return {"logits": s["logits"], "token": s["token"]}
    dec = s["dec"]
    if kind == "step":
        dec.token.copy_(s["tokens"])
        dec.reset(s["pos"])
        first, last = s["pos"], s["pos"] + 1
    else:
        dec.prefill(s["tokens"])
        dec.token.copy_(dec.token_out)
        first, last = 0, s["tokens"].numel() + 1
    dec.enqueue_step(logits=s["logits"], feed_back=False)
    return {"logits": s["logits"], "token": dec.token_out, "x": dec.x,
            "cache": dec.cache[:, first:last].view(torch.bfloat16)}


# ---------------------------------------------------------------- work, tolerance

def _expert_bytes(distinct):
    return distinct * 3 * _H * _I * 2 + 3 * _H * _SI * 2


def _distinct(tokens, skew=0.0):
    """Experts that `tokens` tokens select: the mean of eight draws of the
    logits prepare() makes (weights of std 0.02 against normed states), under
    a Zipf(skew) prior."""
    g = torch.Generator().manual_seed(tokens)
    bias = -skew * (torch.arange(_E) + 1.0).log()
    n = 0
    for _ in range(8):
        z = _STD * math.sqrt(_H) * torch.randn((tokens, _E), generator=g) + bias
        n += z.topk(_K, dim=1).indices.unique().numel()
    return n / 8


_MOE_MAC = 3 * _H * (_K * _I + _SI)             # one token's experts
_ATTN_W = _QKV * _H + _HEADS * (_NOPE + _V) * _LORA + _H * _HEADS * _V


def work(case):
    kind = case["kind"]
    t = case.get("tokens", 1)
    if kind == "route":
        return {"bytes": _E * _H * 2 + t * (_H * 4 + _E * 4 + _K * 8), "flops": 2 * t * _E * _H}
    if kind == "layer":
        return {"bytes": _expert_bytes(_K) + _E * _H * 2, "flops": 2 * _MOE_MAC}
    if kind == "grouped":
        return {"bytes": _expert_bytes(_distinct(t, 1.1)) + t * (2 * _H * 2 + _K * 8),
                "flops": 2 * t * _MOE_MAC}
    if kind == "moe":
        return {"bytes": _expert_bytes(_distinct(t)) + _E * _H * 2 + t * (_H * 6 + _K * 8),
                "flops": 2 * t * (_MOE_MAC + _E * _H)}
    if kind == "attn":
        n = case["pos"] + 1
        return {"bytes": _ATTN_W * 2 + n * _ROW * 2,
                "flops": 2 * (_ATTN_W + _HEADS * n * (_ROW + _LORA))}
    if kind == "dense":
        return {"bytes": 3 * _DENSE * _H * 2, "flops": 2 * 3 * _DENSE * _H}
    if kind == "lm_head":
        return {"bytes": _VOCAB * _H * 2 + _VOCAB * 4, "flops": 2 * _VOCAB * _H}
    head = _VOCAB * _H
    one = _ATTN_W * _LAYERS + (_LAYERS - 1) * (_MOE_MAC + _E * _H) + 3 * _DENSE * _H
    pos = case["pos"] if kind == "step" else t
    step = {"bytes": 2 * (one + head) + _LAYERS * (pos + 1) * _ROW * 2,
            "flops": 2 * (one + head + _LAYERS * _HEADS * (pos + 1) * (_ROW + _LORA))}
    if kind == "step":
        return step
    # the prompt: every weight it touches once, each token's arithmetic, the
    # cache written once; the head once, for the last token
    weights = 2 * (_ATTN_W * _LAYERS + 3 * _DENSE * _H + head) + \
        (_LAYERS - 1) * (_expert_bytes(_distinct(t)) + _E * _H * 2)
    pairs = t * (t + 1) // 2
    return {"bytes": step["bytes"] + weights + _LAYERS * t * _ROW * 2,
            "flops": step["flops"] + 2 * (t * one + head +
                                          _LAYERS * pairs * _HEADS * (_ROW + _LORA))}


def tolerance(case):
    """About four times what this arithmetic with fp32 sums is off from its
    64-bit evaluation, both in plain torch: logits 1.8e-7 (max 9.5e-7); single
    layers 8.7e-5 (one bf16 rounding that falls the other way in 2048 values;
    max one bf16 step, 2^-8); grouped experts 3.2e-4 (max 0.014); the whole
    model 0.037 (27 layers of bf16 roundings), held to 0.03. `differ`: ties of
    the routing and the argmax."""
    kind = case["kind"]
    if kind == "route":
        return {"rel": 1e-6, "max": 4e-6, "differ": 0.01}
    if kind in ("step", "prompt"):
        return {"rel": 0.03, "max": 0.7, "differ": 0.01}
    if kind in ("grouped", "moe"):
        return {"rel": 1.3e-3, "max": 0.06, "differ": 0.01}
    return {"rel": 4e-4, "max": 0.016, "differ": 0.01}


# ---------------------------------------------------------------- 64-bit values

def _bf(t):
    """Rounded to fp32, then to bf16 (nearest even), widened again."""
    return t.float().bfloat16().to(t.dtype)


def _mm(x, w, dt):
    """x @ w^T in dtype dt, x [T][K], w bf16 [N][K], in blocks of rows."""
    out = torch.empty((x.shape[0], w.shape[0]), dtype=dt, device=x.device)
    for a in range(0, w.shape[0], 8192):
        out[:, a: a + 8192] = x.to(dt) @ w[a: a + 8192].to(dt).T
    return out


def _rms(x, gamma, dt):
    ms = x.double().square().mean(-1, keepdim=True).float() + torch.tensor(_D.rms_eps)
    inv = (1.0 / ms.double().sqrt().float().double()).float()
    return _bf(_bf(x.float() * inv) * gamma.float()).to(dt)


def _route(router, x, dt, bias=None):
    logits = _mm(x.to(dt), router.view(_E, _H), dt).float()
    z = logits if bias is None else logits + bias
    p = torch.softmax(z.double(), -1).float()
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    return logits, order.indices[:, :_K], order.values[:, :_K] * _D.routed_scaling


def _mlp(x, w, inter, dt):
    gu = _bf(_mm(x, w[: 2 * inter * _H].view(2 * inter, _H), dt))
    g, u = gu[:, 0::2], gu[:, 1::2]
    s = _bf((g.double() / (1.0 + torch.exp(-g.double()))).to(dt))
    return _bf(_mm(_bf(s * u), w[2 * inter * _H: 3 * inter * _H].view(_H, inter), dt))


def _experts(x, ids, w, experts, shared, dt):
    parts = torch.zeros((x.shape[0], _K, _H), dtype=dt, device=x.device)
    for e in ids.unique().tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        y = _mlp(x[t], experts[e * _D.expert_stride: (e + 1) * _D.expert_stride], _I, dt)
        parts[t, k] = _bf(w[t, k].to(dt)[:, None] * y)
    return _bf(_bf(parts.sum(1)) + _mlp(x, shared, _SI, dt))


def _ffn(x, get, layer, dt):
    """The FFN half of a layer on residual rows x [T][H]."""
    xn = _rms(x, get(f"L{layer}.norm_post"), dt)
    if layer == 0:
        out = _mlp(xn, get("L0.dense"), _DENSE, dt)
        return out, _bf(x.to(dt) + out), None, None
    _, ids, w = _route(get(f"L{layer}.router"), xn, dt)
    out = _experts(xn, ids, w, get(f"L{layer}.experts"), get(f"L{layer}.shared"), dt)
    return out, _bf(x.to(dt) + out), ids, w


def _rotate(v, cos, sin):
    v = v.float()
    y = torch.cat([v[..., 0::2], v[..., 1::2]], -1)
    r = torch.cat([-y[..., _ROPE // 2:], y[..., : _ROPE // 2]], -1)
    return _bf(y * cos + r * sin)


def _attn(x, get, layer, cache, p0, cos, sin, dt):
    """The attention half on rows x [T][H] at positions p0 ..; fills cache."""
    T = x.shape[0]
    xn = _rms(x, get(f"L{layer}.norm_in"), dt)
    qkv = _bf(_mm(xn, get(f"L{layer}.qkv").view(_QKV, _H), dt))
    q = qkv[:, : _HEADS * (_NOPE + _ROPE)].view(T, _HEADS, _NOPE + _ROPE)
    kv = qkv[:, _HEADS * (_NOPE + _ROPE):]
    c, s = cos[p0: p0 + T], sin[p0: p0 + T]
    cache[p0: p0 + T, :_LORA] = _rms(kv[:, :_LORA], get(f"L{layer}.kv_a_norm"), dt).to(cache.dtype)
    cache[p0: p0 + T, _LORA:] = _rotate(kv[:, _LORA:], c, s).to(cache.dtype)
    q_pe = _rotate(q[:, :, _NOPE:], c[:, None], s[:, None]).to(dt)
    kvb = get(f"L{layer}.kv_b").view(_HEADS, _NOPE + _V, _LORA).to(dt)
    rows = cache[: p0 + T].to(dt)
    m = 0.1 * 0.707 * math.log(40.0) + 1.0
    scale = (_NOPE + _ROPE) ** -0.5 * m * m
    later = torch.arange(p0 + T, device=x.device) > torch.arange(p0, p0 + T, device=x.device)[:, None]
    out = torch.empty((T, _HEADS, _V), dtype=dt, device=x.device)
    for h in range(_HEADS):
        q_c = (q[:, h, :_NOPE].to(dt) @ kvb[h, :_NOPE]).float().to(dt)
        sc = (torch.cat([q_c, q_pe[:, h]], -1) @ rows.T.contiguous()) * scale
        pr = torch.softmax(sc.masked_fill(later, -math.inf), -1)
        o_c = (pr @ rows[:, :_LORA].contiguous()).float().to(dt)
        out[:, h] = _bf(o_c @ kvb[h, _NOPE:].T.contiguous())
    o = _bf(_mm(out.view(T, _HEADS * _V), get(f"L{layer}.o_proj").view(_H, _HEADS * _V), dt))
    return _bf(x.to(dt) + o)


def _head(x, get, dt):
    logits = _bf(_mm(_rms(x, get("final_norm"), dt), get("lm_head").view(_VOCAB, _H), dt))
    return logits, logits.max(-1, keepdim=True).values.eq(logits).to(torch.int8).argmax(-1)


def _model(tokens, p0, get, caches, cos, sin, dt):
    x = get("embed").view(_VOCAB, _H)[tokens.long()].to(dt)
    for i in range(_LAYERS):
        x = _attn(x, get, i, caches[i], p0, cos, sin, dt)
        x = _ffn(x, get, i, dt)[1]
    logits, best = _head(x[-1:], get, dt)
    return x, logits[0], best


def _evaluate(case, seed, dt):
    kind, s = case["kind"], _inputs(case, seed)

    def get(name):
        return _tensor(s["blob"], s["lay"], name)

    if kind == "route":
        return _route(get("L1.router"), s["x"], dt)
    if kind == "grouped":
        return _experts(s["x"].to(dt), s["ids"], s["w"], get("L1.experts"), get("L1.shared"), dt)
    if kind == "moe":
        logits, ids, w = _route(get("L1.router"), s["x"], dt)
        out = _experts(s["x"].to(dt), ids, w, get("L1.experts"), get("L1.shared"), dt)
        return {"logits": logits, "ids": ids, "weights": w, "out": out}
    if kind == "layer":
        out, x_out, ids, w = _ffn(s["x"][None], get, 1, dt)
        return {"x_out": x_out[0], "moe_out": out[0], "ids": ids[0], "weights": w[0]}
    if kind == "dense":
        out, x_out, _, _ = _ffn(s["x"][None], get, 0, dt)
        return {"x_out": x_out[0], "mlp_out": out[0]}
    if kind == "lm_head":
        logits, best = _head(s["x"][None], get, dt)
        return {"logits": logits[0], "token": best}
    cos, sin = _tables()
    if kind == "attn":
        x_out = _attn(s["x"][None], get, 0, s["cache"], case["pos"], cos, sin, dt)
        return {"x_out": x_out[0], "row": s["cache"][case["pos"]].to(dt)}
    caches = torch.zeros((_LAYERS, _MAX_POS, _ROW), dtype=torch.bfloat16, device=_DEV)
    tokens, first, pos = s["tokens"], 0, s["tokens"].numel()
    if kind == "step":
        first = pos = case["pos"]
        caches[:, :pos] = s["rows"]
    else:
        _, _, tokens = _model(tokens, 0, get, caches, cos, sin, dt)
    x, logits, best = _model(tokens, pos, get, caches, cos, sin, dt)
    return {"logits": logits, "token": best, "x": x[-1],
            "cache": caches[:, first: pos + 1].to(dt)}


def exact(case, seed):
    return _evaluate(case, seed, torch.float64)
