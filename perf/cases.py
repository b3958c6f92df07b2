"""The work this framework is timed on: its public calls over the sizes they serve.

A case is a dict of plain values whose "kind" names the call:

  linear        `Q4Linear` (fp32 result) or `Q4Weight.matmul` (16-bit result) on
                `rows` activation rows: decode (1 row), speculative verify and
                small batches (2..16), short prompts and whole prompts
  mlp           the SwiGLU `MLP` module over packed projections
  attn_decode   `attention_decode` over an int8 KV cache, one query row a sequence
  attn_layer    the `Attention` module (packed projections, RoPE, int8 append,
                attention) over `new` tokens behind `cached` ones
  step          one decode step of the whole decoder, replayed from its graph
  prefill       a whole prompt through the decoder

Weights are int4 with fp16 group scales, quantized round-to-nearest from normal
draws; activations are normal with per-channel scales, as after a norm layer.
`exact` restates each call in 64 bits with plain torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from siliconfer_amd.kernels.attention import attention_decode
from siliconfer_amd.kernels.q4 import Q4Weight
from siliconfer_amd.model.config import ModelConfig
from siliconfer_amd.model.kv_cache import QuantizedKVCache
from siliconfer_amd.model.layers import MLP, Attention, compute_rope_freqs
from siliconfer_amd.model.llama import LayerWeights, LlamaModel
from siliconfer_amd.model.q4_linear import Q4Linear

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed() -> list[dict]:
    return [
        # one decoded token through the 0.5B up projection: the smallest call, where
        # latency counts
        dict(name="decode_row_small", kind="linear", rows=1, n=4864, k=896, group=64, asym=False,
             dtype="f16", out="f32"),
        # one decoded token through a 7B down projection: the weight stream
        dict(name="decode_row_7b", kind="linear", rows=1, n=4096, k=11008, group=128, asym=False,
             dtype="f16", out="same"),
        # eight verify rows through an 8B up projection with zero-points
        dict(name="verify_rows_8b", kind="linear", rows=8, n=14336, k=4096, group=64, asym=True,
             dtype="bf16", out="f32"),
        # a short prompt (ragged) through a 7B up projection
        dict(name="short_prompt_7b", kind="linear", rows=37, n=11008, k=4096, group=128, asym=False,
             dtype="f16", out="same"),
        # a 512-token prompt through the 0.5B up projection with zero-points
        dict(name="prompt_small", kind="linear", rows=512, n=4864, k=896, group=64, asym=True,
             dtype="bf16", out="same"),
        # a 2048-token prompt through a 7B down projection
        dict(name="prompt_7b", kind="linear", rows=2048, n=4096, k=11008, group=128, asym=False,
             dtype="bf16", out="same"),
        # a ragged prompt through the 8B MLP module, fp32 activations (the modules' default)
        dict(name="mlp_prompt_8b", kind="mlp", rows=333, hidden=4096, inter=14336, group=128,
             asym=False, dtype="f32"),
        # decode attention of the 0.5B geometry over 4096 cached tokens
        dict(name="attn_decode_small", kind="attn_decode", batch=1, heads=14, kv_heads=2, dim=64,
             cached=4096, dtype="f16"),
        # batched decode attention of the 8B geometry over long ragged caches
        dict(name="attn_decode_long", kind="attn_decode", batch=4, heads=32, kv_heads=8, dim=128,
             cached=8191, dtype="bf16"),
        # the 8B attention layer over a ragged prompt chunk behind a cached prefix
        dict(name="attn_layer_prompt", kind="attn_layer", hidden=4096, heads=32, kv_heads=8,
             dim=128, new=1500, cached=300, group=128, dtype="f32"),
        # one decode step of the whole 0.5B decoder after a 512-token prompt
        dict(name="decoder_step", kind="step", cached=512, dtype="f16"),
        # a 512-token prompt through the whole 0.5B decoder
        dict(name="decoder_prompt", kind="prefill", rows=512, dtype="f16"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear"] * 5 + ["mlp", "attn_decode", "attn_decode", "attn_layer",
                                        "attn_layer", "step", "prefill"])
    group = rng.choice([64, 128])
    dtype = rng.choice(["f32", "f16", "bf16"])
    if kind == "linear":
        rows = _log_int(rng, 1, 2048)
        n = _log_int(rng, 896, 14336)
        k = group * max(1, _log_int(rng, 896, 14336) // group)
        if rng.random() < 0.7:  # most layers are multiples of 64 wide, some are ragged
            n = 64 * max(1, n // 64)
        cap = 2048 * 4096 * 11008 // (2 if dtype == "f32" else 1)
        rows = max(1, min(rows, cap // (n * k)))
        return dict(kind=kind, rows=rows, n=n, k=k, group=group, asym=rng.random() < 0.5,
                    dtype=dtype, out=rng.choice(["f32", "same"]))
    if kind == "mlp":
        hidden = group * (_log_int(rng, 896, 4096) // group)
        inter = group * (_log_int(rng, 2432, 14336) // group)
        return dict(kind=kind, rows=_log_int(rng, 1, 333), hidden=hidden, inter=inter, group=group,
                    asym=rng.random() < 0.5, dtype=dtype)
    if kind == "attn_decode":
        heads, kv_heads, dim = rng.choice([(14, 2, 64), (32, 8, 128), (32, 32, 128)])
        batch = rng.choice([1, 1, 2, 4])
        cached = _log_int(rng, 100, 16384)
        cached = min(cached, 4 * 8 * 8191 // (batch * kv_heads))
        return dict(kind=kind, batch=batch, heads=heads, kv_heads=kv_heads, dim=dim, cached=cached,
                    dtype=dtype)
    if kind == "attn_layer":
        hidden, heads, kv_heads, dim = rng.choice([(896, 14, 2, 64), (4096, 32, 8, 128),
                                                   (4096, 32, 32, 128)])
        new = _log_int(rng, 1, 1500 if kv_heads <= 8 else 1000)
        return dict(kind=kind, hidden=hidden, heads=heads, kv_heads=kv_heads, dim=dim, new=new,
                    cached=rng.choice([0, _log_int(rng, 20, 300)]), group=group, dtype=dtype)
    if kind == "step":
        return dict(kind=kind, cached=_log_int(rng, 32, 1000), dtype=dtype)
    return dict(kind=kind, rows=_log_int(rng, 16, 512), dtype=dtype)


# ---------------------------------------------------------------- inputs
_DEV = "cuda"


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _randn(gen, *shape) -> torch.Tensor:
    return torch.randn(*shape, generator=gen, device=_DEV, dtype=torch.float32)


def _activations(gen, rows: int, width: int) -> torch.Tensor:
    return _randn(gen, rows, width) * torch.exp(0.5 * _randn(gen, width))


def _quantize(W: torch.Tensor, group: int, asym: bool):
    """Round-to-nearest int4: (codes int8 [N, K], scales fp16-valued fp32 [N, G], zeros or None)."""
    N, K = W.shape
    g = W.reshape(N, K // group, group)
    if asym:
        lo, hi = g.amin(-1, keepdim=True).clamp(max=0.0), g.amax(-1, keepdim=True).clamp(min=0.0)
        s = ((hi - lo) / 15.0).clamp(min=1e-6)
        z = torch.round(-lo / s).clamp(0, 15)
        q = (torch.round(g / s) + z).clamp(0, 15)
    else:
        s = (g.abs().amax(-1, keepdim=True) / 7.0).clamp(min=1e-6)
        z = None
        q = torch.round(g / s).clamp(-8, 7)
    return (q.reshape(N, K).to(torch.int8), s[..., 0].to(torch.float16).float(),
            None if z is None else z[..., 0].contiguous())


def _pack(q: torch.Tensor) -> torch.Tensor:
    u = q.view(torch.uint8) & 0x0F
    return (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()


def _weight(gen, n: int, k: int, group: int, asym: bool):
    return _quantize(_randn(gen, n, k) * 0.02, group, asym)


def _dense64(weight, group: int) -> torch.Tensor:
    q, s, z = weight
    N, K = q.shape
    w = q.reshape(N, K // group, group).double()
    if z is not None:
        w = w - z.double()[..., None]
    return (w * s.double()[..., None]).reshape(N, K)


def _q4linear(weight, group: int) -> Q4Linear:
    q, s, z = weight
    return Q4Linear(_pack(q), s, z, None, group)


def _linear_inputs(case: dict, seed: int):
    gen = _gen(seed)
    w = _weight(gen, case["n"], case["k"], case["group"], case["asym"])
    return w, _activations(gen, case["rows"], case["k"]).to(_DTYPES[case["dtype"]])


def _mlp_inputs(case: dict, seed: int):
    gen = _gen(seed)
    H, I, g, a = case["hidden"], case["inter"], case["group"], case["asym"]
    ws = [_weight(gen, I, H, g, a), _weight(gen, I, H, g, a), _weight(gen, H, I, g, a)]
    return ws, _activations(gen, case["rows"], H).to(_DTYPES[case["dtype"]])


def _decode_inputs(case: dict, seed: int):
    gen = _gen(seed)
    B, H, KVH, D, T = (case[x] for x in ("batch", "heads", "kv_heads", "dim", "cached"))
    dt = _DTYPES[case["dtype"]]
    # keys share a direction per head, so that scores spread over several units as trained ones do
    k = (_randn(gen, B, KVH, T, D) + _randn(gen, B, KVH, 1, D)).to(dt)
    v = _randn(gen, B, KVH, T, D).to(dt)
    q = (1.5 * _randn(gen, B, H, D)).to(dt)
    return q, k, v


def _layer_config(case: dict) -> ModelConfig:
    return ModelConfig(hidden_size=case["hidden"], intermediate_size=0, num_hidden_layers=1,
                       num_attention_heads=case["heads"], num_key_value_heads=case["kv_heads"],
                       head_dim=case["dim"], vocab_size=0, rope_theta=500000.0)


def _layer_inputs(case: dict, seed: int):
    gen = _gen(seed)
    Hd, H, KVH, D, g = (case[x] for x in ("hidden", "heads", "kv_heads", "dim", "group"))
    ws = [_weight(gen, H * D, Hd, g, False), _weight(gen, KVH * D, Hd, g, False),
          _weight(gen, KVH * D, Hd, g, False), _weight(gen, Hd, H * D, g, False)]
    x = _activations(gen, case["new"], Hd).to(_DTYPES[case["dtype"]])[None]
    k = _randn(gen, 1, KVH, case["cached"], D)
    v = _randn(gen, 1, KVH, case["cached"], D)
    return ws, x, k, v


def _decoder_inputs(case: dict, seed: int, count: int):
    """The 0.5B geometry with random weights, `count` prompt ids and one more token."""
    c = ModelConfig.qwen25_05b()
    gen = _gen(seed)
    H, I, D, Hq, KVH = (c.hidden_size, c.intermediate_size, c.head_dim, c.num_attention_heads,
                        c.num_key_value_heads)
    layers = []
    for _ in range(c.num_hidden_layers):
        qkv = _weight(gen, (Hq + 2 * KVH) * D, H, 64, False)
        layers.append(dict(qkv=qkv, bias=_randn(gen, (Hq + 2 * KVH) * D) * 0.02,
                           o=_weight(gen, H, Hq * D, 64, False),
                           gate_up=_weight(gen, 2 * I, H, 64, False),
                           down=_weight(gen, H, I, 64, False),
                           w_in=1.0 + 0.1 * _randn(gen, H), w_post=1.0 + 0.1 * _randn(gen, H)))
    embed = (_randn(gen, c.vocab_size, H) * 0.02).to(torch.bfloat16)
    norm = 1.0 + 0.1 * _randn(gen, H)
    ids = torch.randint(0, c.vocab_size, (count + 1,), generator=gen, device=_DEV)
    return c, layers, embed, norm, ids


def _decoder(case: dict, seed: int, count: int):
    c, layers, embed, norm, ids = _decoder_inputs(case, seed, count)

    def q4(w):
        return Q4Weight(_pack(w[0]), w[1], w[2], 64)

    lw = [LayerWeights(q4(d["qkv"]), d["bias"], q4(d["o"]), q4(d["gate_up"]), q4(d["down"]),
                       d["w_in"], d["w_post"]) for d in layers]
    model = LlamaModel(c, lw, embed, norm, 64, 1024, act_dtype=_DTYPES[case["dtype"]])
    return model, ids


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        if case["out"] == "same":
            return dict(kind=kind, call=Q4Weight(_pack(w[0]), w[1], w[2], case["group"]).matmul, x=x)
        return dict(kind=kind, call=_q4linear(w, case["group"]), x=x)
    if kind == "mlp":
        ws, x = _mlp_inputs(case, seed)
        # the module's own dense layers are replaced by packed ones: make them small
        mod = MLP(ModelConfig(hidden_size=8, intermediate_size=8), device=_DEV)
        mod.gate_proj, mod.up_proj, mod.down_proj = (_q4linear(w, case["group"]) for w in ws)
        return dict(kind=kind, call=mod, x=x)
    if kind == "attn_decode":
        q, k, v = _decode_inputs(case, seed)
        cache = QuantizedKVCache(capacity=case["cached"] + 64)
        cache.append(k, v)
        return dict(kind=kind, q=q, cache=cache)
    if kind == "attn_layer":
        ws, x, k, v = _layer_inputs(case, seed)
        c = _layer_config(case)
        mod = Attention(c, compute_rope_freqs(c), device=_DEV)
        mod.q_proj, mod.k_proj, mod.v_proj, mod.o_proj = (_q4linear(w, case["group"]) for w in ws)
        cache = QuantizedKVCache(capacity=2048)
        if case["cached"]:
            cache.append(k, v)
        return dict(kind=kind, call=mod, x=x, cache=cache, cached=case["cached"])
    if kind == "step":
        model, ids = _decoder(case, seed, case["cached"])
        model.capture(logits=True)
        model.prefill(ids[:-1].cpu().numpy())
        return dict(kind=kind, model=model, token=ids[-1:].to(torch.int32), cached=case["cached"])
    model, ids = _decoder(case, seed, case["rows"])
    return dict(kind=kind, model=model, ids=ids[:-1].cpu().numpy())


def run(state: dict):
    kind = state["kind"]
    if kind in ("linear", "mlp"):
        return state["call"](state["x"])
    if kind == "attn_decode":
        c = state["cache"]
        return attention_decode(state["q"], *c.buffers(), T=c.length())
    if kind == "attn_layer":
        c = state["cache"]
        c.trim(state["cached"])  # back to the prefix: the call appends its own tokens
        y, c = state["call"](state["x"], c)
        return y, c.q_k, c.q_v
    model = state["model"]
    if kind == "step":
        model.set_position(state["cached"])
        model.token.copy_(state["token"])
        model.replay(1)
        return model.logits
    model.reset()
    model.prefill(state["ids"])
    return model.logits


# ---------------------------------------------------------------- work
def _q4_bytes(n: int, k: int, group: int, asym: bool) -> float:
    return n * k / 2 + n * (k // group) * (2.5 if asym else 2.0)


_05B = dict(layers=24, hidden=896, inter=4864, qkv=1152, heads=14, kv_heads=2, dim=64, vocab=151936)


def _decoder_weights() -> tuple[float, float]:
    """(bytes, weight count) of the 0.5B decoder's layers."""
    m = _05B
    mats = [(m["qkv"], m["hidden"]), (m["hidden"], m["heads"] * m["dim"]),
            (2 * m["inter"], m["hidden"]), (m["hidden"], m["inter"])]
    return (m["layers"] * sum(_q4_bytes(n, k, 64, False) for n, k in mats),
            m["layers"] * sum(n * k for n, k in mats))


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        r, n, k = case["rows"], case["n"], case["k"]
        e = _SIZE[case["dtype"]]
        return {"bytes": _q4_bytes(n, k, case["group"], case["asym"]) + r * k * e
                + r * n * (e if case["out"] == "same" else 4), "flops": 2.0 * r * n * k}
    if kind == "mlp":
        r, h, i = case["rows"], case["hidden"], case["inter"]
        w = 2 * _q4_bytes(i, h, case["group"], case["asym"]) + _q4_bytes(h, i, case["group"], case["asym"])
        return {"bytes": w + r * h * (_SIZE[case["dtype"]] + 4), "flops": 6.0 * r * h * i}
    if kind == "attn_decode":
        b, h, kv, d, t = (case[x] for x in ("batch", "heads", "kv_heads", "dim", "cached"))
        return {"bytes": 2.0 * b * kv * t * (d + 2) + b * h * d * (_SIZE[case["dtype"]] + 4),
                "flops": 4.0 * b * h * t * d}
    if kind == "attn_layer":
        hd, h, kv, d, t, t0 = (case[x] for x in ("hidden", "heads", "kv_heads", "dim", "new", "cached"))
        mats = [(h * d, hd), (kv * d, hd), (kv * d, hd), (hd, h * d)]
        pairs = t * (t0 + (t + 1) / 2.0)
        return {"bytes": sum(_q4_bytes(n, k, case["group"], False) for n, k in mats)
                + t * hd * (_SIZE[case["dtype"]] + 4) + 2.0 * kv * (t0 + t) * (d + 2),
                "flops": sum(2.0 * t * n * k for n, k in mats) + 4.0 * h * d * pairs}
    m = _05B
    wb, wn = _decoder_weights()
    kv_row = 2.0 * m["layers"] * m["kv_heads"] * (m["dim"] + 2)
    head = 2.0 * m["vocab"] * m["hidden"]
    if kind == "step":
        t = case["cached"] + 1
        return {"bytes": wb + head + kv_row * t + 4.0 * m["vocab"],
                "flops": 2 * wn + head + 4.0 * m["layers"] * m["heads"] * m["dim"] * t}
    t = case["rows"]
    return {"bytes": wb + head + kv_row * t + 2.0 * t * m["hidden"] + 4.0 * m["vocab"],
            "flops": 2 * wn * t + head + 4.0 * m["layers"] * m["heads"] * m["dim"] * t * (t + 1) / 2.0}


def tolerance(case: dict):
    """About four times the measured distance from `exact` (2-norm)."""
    kind, dt = case["kind"], case["dtype"]
    if kind == "linear":
        if case["out"] == "same" and dt != "f32":
            return {"rel": 7e-3 if dt == "bf16" else 1e-3}  # the result's own rounding
        return {"rel": 2e-5}  # 32-bit sums; fp32 activations as two 16-bit halves
    if kind == "mlp":
        # three such products, the second on 32-bit results of the first
        return {"rel": 1e-4}
    if kind == "attn_decode":
        return {"rel": 2e-5}
    if kind == "attn_layer":
        # a 32-bit difference ahead of the int8 rounding moves a code by one here and there
        return {"rel": 4e-3, "differ": 5e-3}
    return {"rel": 2e-2}  # 24 layers of 16-bit activations and int8 codes


# ---------------------------------------------------------------- 64-bit restatement
def _quant_kv(x: torch.Tensor):
    """int8 codes (as doubles) and fp16-valued scales of [..., D] vectors, in 32 bits as the cache
    defines them."""
    x = x.float()
    s = x.abs().amax(-1, keepdim=True)
    s = s / torch.full_like(s, 127.0)
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.round(x / s).clamp(-128, 127).double(), s.half().double()


def _rope64(x: torch.Tensor, start: int, theta: float) -> torch.Tensor:
    """Rotate-half RoPE of [T, heads, D] (fp32 angles, as the tables hold them)."""
    D = x.shape[-1]
    f = (1.0 / (np.float32(theta) ** (np.arange(0, D, 2, dtype=np.float32) / np.float32(D)))).astype(np.float32)
    ang = np.outer(np.arange(start, start + x.shape[0], dtype=np.float32), f).astype(np.float32)
    c = torch.from_numpy(np.cos(ang)).double().to(x.device)[:, None]
    s = torch.from_numpy(np.sin(ang)).double().to(x.device)[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend64(q, k, v, t0: int) -> torch.Tensor:
    """Causal attention of q [T, H, D] at positions t0.. over k, v [KVH, t0 + T, D]."""
    T, H, D = q.shape
    out = torch.empty_like(q)
    mask = (torch.arange(k.shape[1], device=q.device)[None, :]
            > torch.arange(T, device=q.device)[:, None] + t0)
    for h in range(H):
        j = h // (H // k.shape[0])
        s = (q[:, h] @ k[j].t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), dim=-1) @ v[j]
    return out


def _norm64(x, w, eps: float):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _decoder64(case: dict, seed: int, count: int, with_token: bool) -> torch.Tensor:
    c, layers, embed, norm, ids = _decoder_inputs(case, seed, count)
    ids = ids if with_token else ids[:-1]
    T, Hq, KVH, D = ids.numel(), c.num_attention_heads, c.num_key_value_heads, c.head_dim
    h = embed[ids].double()
    for L in layers:
        x = _norm64(h, L["w_in"], c.rms_norm_eps)
        qkv = x @ _dense64(L["qkv"], 64).t() + L["bias"].double()
        q, k, v = qkv.reshape(T, Hq + 2 * KVH, D).split([Hq, KVH, KVH], dim=1)
        q, k = _rope64(q, 0, c.rope_theta), _rope64(k, 0, c.rope_theta)
        kq, ks = _quant_kv(k.transpose(0, 1))
        vq, vs = _quant_kv(v.transpose(0, 1))
        a = _attend64(q, kq * ks, vq * vs, 0).reshape(T, Hq * D)
        h = h + a @ _dense64(L["o"], 64).t()
        g, u = (_norm64(h, L["w_post"], c.rms_norm_eps) @ _dense64(L["gate_up"], 64).t()).chunk(2, dim=1)
        h = h + (torch.nn.functional.silu(g) * u) @ _dense64(L["down"], 64).t()
    return embed.double() @ _norm64(h[-1], norm, c.rms_norm_eps)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        return x.double() @ _dense64(w, case["group"]).t()
    if kind == "mlp":
        ws, x = _mlp_inputs(case, seed)
        g, u, d = (_dense64(w, case["group"]).t() for w in ws)
        x = x.double()
        return (torch.nn.functional.silu(x @ g) * (x @ u)) @ d
    if kind == "attn_decode":
        q, k, v = _decode_inputs(case, seed)
        kq, ks = _quant_kv(k)
        vq, vs = _quant_kv(v)
        T = case["cached"]
        return torch.stack([_attend64(q[b:b + 1].double(), kq[b] * ks[b], vq[b] * vs[b], T - 1)[0]
                            for b in range(case["batch"])])
    if kind == "attn_layer":
        ws, x, k0, v0 = _layer_inputs(case, seed)
        T, H, KVH, D, t0 = case["new"], case["heads"], case["kv_heads"], case["dim"], case["cached"]
        wq, wk, wv, wo = (_dense64(w, case["group"]).t() for w in ws)
        x = x[0].double()
        q = _rope64((x @ wq).reshape(T, H, D), t0, 500000.0)
        k = _rope64((x @ wk).reshape(T, KVH, D), t0, 500000.0).transpose(0, 1)
        v = (x @ wv).reshape(T, KVH, D).transpose(0, 1)
        (kq, ks), (vq, vs) = (_quant_kv(torch.cat([a[0].double(), b], dim=1)) for a, b in ((k0, k), (v0, v)))
        y = _attend64(q, kq * ks, vq * vs, t0).reshape(T, H * D) @ wo
        return y[None], kq.to(torch.int8)[None], vq.to(torch.int8)[None]
    if kind == "step":
        return _decoder64(case, seed, case["cached"], True)
    return _decoder64(case, seed, case["rows"], False)
