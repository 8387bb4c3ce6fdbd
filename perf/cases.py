"""Performance cases: what training and serving programs ask of this package, at sizes from the smallest
call to the largest.

The shapes are Qwen3-8B's (hidden 4096, intermediate 12288, 32 query and 8 key/value heads of 128,
vocabulary 151936) and the four-layer configuration of the tiny training step; weights are random.  A case
is a dict with a ``kind`` and its sizes; ``prepare`` / ``run`` / ``work`` / ``tolerance`` / ``exact``
dispatch on the kind.  Most kinds are one layer or one operator family; ``prefill`` and ``decode`` are whole
model calls over a few layers (every layer costs the same) and return logits and the key/value cache.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3-triton_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

H, I, HQ, HKV, D, V = 4096, 12288, 32, 8, 128, 151936   # Qwen3-8B
TH, TI, THQ, THKV, TD, TV, TL = 256, 688, 8, 2, 32, 4096, 4   # the tiny training configuration
THETA, EPS = 1e6, 1e-6
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


# ------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # One optimizer step's forward + backward of the four-layer tiny model: the smallest whole training
        # call, where the number of launches and the host's share count.
        {"name": "tiny_step_b2_s128", "kind": "tiny", "batch": 2, "seq": 128, "dtype": "bf16"},
        # Fine-tuning on one unpadded sample: a decoder layer at a ragged token count.
        {"name": "layer_b1_s333", "kind": "layer", "batch": 1, "seq": 333},
        # The training step the benchmark reports: a decoder layer at 8192 tokens.
        {"name": "layer_b4_s2048", "kind": "layer", "batch": 4, "seq": 2048},
        # Attention alone, forward + backward: a ragged middle-sized batch in fp16 and a long context in bf16.
        {"name": "attention_b3_s1000_f16", "kind": "attention", "batch": 3, "seq": 1000, "dtype": "f16"},
        {"name": "attention_b1_s8192", "kind": "attention", "batch": 1, "seq": 8192, "dtype": "bf16"},
        # The fused LM head + loss of the training step, forward + backward (the largest case).
        {"name": "lm_head_b4_s2048", "kind": "lm_head", "batch": 4, "seq": 2048},
        # The bandwidth-bound operators of a layer, forward + backward: RMSNorm, Q/K norm + RoPE, SwiGLU.
        {"name": "pointwise_t8192", "kind": "pointwise", "batch": 4, "seq": 2048},
        # Serving, first token: a short prompt (65 tokens, the request of the inference benchmark), and a long
        # ragged one.
        {"name": "prefill_b1_s65", "kind": "prefill", "batch": 1, "seq": 65},
        {"name": "prefill_b1_s1500", "kind": "prefill", "batch": 1, "seq": 1500},
        # Serving, next token: one request, a small batch, and a batch of many users.
        {"name": "decode_b1_t2048", "kind": "decode", "batch": 1, "context": 2048},
        {"name": "decode_b8_t1024", "kind": "decode", "batch": 8, "context": 1024},
        {"name": "decode_b32_t300", "kind": "decode", "batch": 32, "context": 300},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tiny", "layer", "attention", "lm_head", "pointwise", "prefill", "decode"])
    if kind == "tiny":
        return {"kind": kind, "batch": rng.randint(1, 4), "seq": _log_int(rng, 17, 512),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "attention":
        b = rng.randint(1, 4)
        return {"kind": kind, "batch": b, "seq": _log_int(rng, 64, 8192 // b), "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "decode":
        return {"kind": kind, "batch": _log_int(rng, 1, 40), "context": _log_int(rng, 40, 4096)}
    b = rng.randint(1, 4)
    return {"kind": kind, "batch": b, "seq": _log_int(rng, 17 if kind == "prefill" else 64, 8192 // b)}


# ------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape, dtype=torch.bfloat16, std=1.0):
    t = torch.empty(shape, device="cuda", dtype=dtype)
    return t.normal_(0.0, std, generator=gen)


def _norm_weight(gen, n, dtype=torch.bfloat16):
    return (1 + 0.1 * torch.randn(n, device="cuda", generator=gen)).to(dtype)


def _config(**kw):
    from transformers import Qwen3Config
    base = dict(vocab_size=V, hidden_size=H, intermediate_size=I, num_attention_heads=HQ, num_key_value_heads=HKV,
                head_dim=D, rope_theta=THETA, rms_norm_eps=EPS, tie_word_embeddings=False,
                max_position_embeddings=40960, initializer_range=0.02)
    base.update(kw)
    return Qwen3Config(**base)


def _tables(batch, seq, d, dtype):
    from qwen3_triton.kernels.rotary import rotary_tables
    pos = torch.arange(seq, device="cuda").repeat(batch, 1)
    inv = (1.0 / (THETA ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).cuda()
    return rotary_tables(pos, inv, dtype)


def _module_on_gpu(make, gen, dtype):
    """make()'s module with N(0, 0.02) matrices and norm weights near 1, created on the GPU."""
    with torch.device("meta"):
        m = make()
    m = m.to(dtype).to_empty(device="cuda")
    with torch.no_grad():
        for name, p in m.named_parameters():
            p.copy_(_norm_weight(gen, p.numel(), dtype)) if name.endswith("norm.weight") else \
                p.normal_(0.0, 0.02, generator=gen)
    return m


def _labels(gen, batch, seq, vocab):
    labels = torch.randint(0, vocab, (batch, seq), device="cuda", generator=gen)
    drop = torch.rand(batch, seq, device="cuda", generator=gen) < 0.05   # 5 % of the tokens carry no loss
    return torch.where(drop, torch.full_like(labels, -100), labels)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _gen(seed), seed)


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------------------------------ tiny training step
def _tiny_prepare(case, gen, seed):
    from qwen3_triton.configuration import OptimizationOptions
    from qwen3_triton.model import PrecisionQwen3ForCausalLM
    cfg = _config(vocab_size=TV, hidden_size=TH, intermediate_size=TI, num_hidden_layers=TL, num_attention_heads=THQ,
                  num_key_value_heads=THKV, head_dim=TD, max_position_embeddings=4096)
    dt = DTYPES[case["dtype"]]
    m = _module_on_gpu(lambda: PrecisionQwen3ForCausalLM(cfg, OptimizationOptions(), require_8b_shape=False), gen, dt)
    m.model.rotary_emb.inv_freq = (1.0 / (THETA ** (torch.arange(0, TD, 2, dtype=torch.float32) / TD))).cuda()
    return {"kind": "tiny", "model": m, "params": [p for _, p in sorted(m.named_parameters())],
            "ids": torch.randint(0, TV, (case["batch"], case["seq"]), device="cuda", generator=gen)}


def _tiny_run(st):
    out = st["model"](st["ids"], labels=st["ids"])
    grads = torch.autograd.grad(out.loss, st["params"])
    return {"logits": out.logits, "loss": out.loss, "grads": list(grads)}


# ------------------------------------------------------------------------------------------ one decoder layer
def _layer_prepare(case, gen, seed):
    from qwen3_triton.components import DecoderLayer
    from qwen3_triton.configuration import OptimizationOptions
    b, s = case["batch"], case["seq"]
    layer = _module_on_gpu(lambda: DecoderLayer(_config(num_hidden_layers=1), OptimizationOptions()), gen, torch.bfloat16)
    return {"kind": "layer", "layer": layer, "params": [p for _, p in sorted(layer.named_parameters())],
            "x": _randn(gen, b, s, H).requires_grad_(), "dy": _randn(gen, b, s, H),
            "tables": _tables(b, s, D, torch.bfloat16)}


def _layer_run(st):
    y = st["layer"](st["x"], st["tables"])
    grads = torch.autograd.grad(y, [st["x"]] + st["params"], st["dy"])
    return {"y": y, "grads": list(grads)}


# ------------------------------------------------------------------------------------------ attention
def _attention_prepare(case, gen, seed):
    b, s, dt = case["batch"], case["seq"], DTYPES[case["dtype"]]
    q, k = _randn(gen, b, s, HQ, D, dtype=dt), _randn(gen, b, s, HKV, D, dtype=dt)
    v = _randn(gen, b, s, HKV, D, dtype=dt, std=1.28)
    return {"kind": "attention", "qkv": [t.requires_grad_() for t in (q, k, v)], "do": _randn(gen, b, s, HQ, D, dtype=dt)}


def _attention_run(st):
    from qwen3_triton.kernels.attention import causal_attention_bshd
    o = causal_attention_bshd(*st["qkv"])
    return {"o": o, "grads": list(torch.autograd.grad(o, st["qkv"], st["do"]))}


# ------------------------------------------------------------------------------------------ LM head + loss
def _lm_head_prepare(case, gen, seed):
    b, s = case["batch"], case["seq"]
    return {"kind": "lm_head", "x": _randn(gen, b, s, H).requires_grad_(),
            "w": _randn(gen, V, H, std=0.02).requires_grad_(), "labels": _labels(gen, b, s, V)}


def _lm_head_run(st):
    from qwen3_triton.kernels.lm_head_ce import lm_head_cross_entropy
    loss = lm_head_cross_entropy(st["x"], st["w"], st["labels"])
    dx, dw = torch.autograd.grad(loss, [st["x"], st["w"]])
    return {"loss": loss, "dx": dx, "dw": dw}


# ------------------------------------------------------------------------------------------ bandwidth-bound operators
def _pointwise_prepare(case, gen, seed):
    b, s = case["batch"], case["seq"]
    shapes = {"x": (b, s, H), "q": (b, s, HQ, D), "k": (b, s, HKV, D), "g": (b, s, I), "u": (b, s, I)}
    t = {n: _randn(gen, *sh).requires_grad_() for n, sh in shapes.items()}
    up = {n: _randn(gen, *shapes[n]) for n in ("x", "q", "k", "g")}
    w = {n: _norm_weight(gen, k).requires_grad_() for n, k in (("x", H), ("q", D), ("k", D))}
    return {"kind": "pointwise", "t": t, "w": w, "up": up, "tables": _tables(b, s, D, torch.bfloat16)}


def _pointwise_run(st):
    from qwen3_triton.kernels.activation import swiglu
    from qwen3_triton.kernels.norm import rms_norm
    from qwen3_triton.kernels.norm_rope import norm_rope_pair
    t, w, up = st["t"], st["w"], st["up"]
    n = rms_norm(t["x"], w["x"], EPS)
    q, k = norm_rope_pair(t["q"], t["k"], w["q"], w["k"], *st["tables"], EPS)
    y = swiglu(t["g"], t["u"])
    dx = torch.autograd.grad(n, [t["x"], w["x"]], up["x"])
    dqk = torch.autograd.grad([q, k], [t["q"], t["k"], w["q"], w["k"]], [up["q"], up["k"]])
    dgu = torch.autograd.grad(y, [t["g"], t["u"]], up["g"])
    return {"out": [n, q, k, y], "grads": [*dx, *dqk, *dgu]}


# ------------------------------------------------------------------------------------------ serving
PREFILL_LAYERS, DECODE_LAYERS = 2, 4


def _model(seed, layers):
    from qwen3_triton.inference import TritonQwen3Inference
    return TritonQwen3Inference.random_init(_config(num_hidden_layers=layers), seed=seed)


def _prefill_prepare(case, gen, seed):
    return {"kind": "prefill", "model": _model(seed, PREFILL_LAYERS),
            "ids": torch.randint(0, V, (case["batch"], case["seq"]), device="cuda", generator=gen)}


def _prefill_run(st):
    out = st["model"](st["ids"])
    return {"logits": out.logits, "keys": out.past_key_values.keys, "values": out.past_key_values.values}


def _decode_prepare(case, gen, seed):
    b, t = case["batch"], case["context"]
    model = _model(seed, DECODE_LAYERS)
    cache = model.new_cache(b, t + 1)
    for k, v in zip(cache.keys, cache.values):   # normed keys have unit scale, values that of a projection
        k.normal_(0.0, 1.0, generator=gen)
        v.normal_(0.0, 1.28, generator=gen)
    return {"kind": "decode", "model": model, "cache": cache, "context": t,
            "ids": torch.randint(0, V, (b, 1), device="cuda", generator=gen)}


def _decode_run(st):
    st["cache"].length = st["context"]   # the next token of the same context
    out = st["model"](st["ids"], past_key_values=st["cache"])
    return {"logits": out.logits, "keys": st["cache"].keys, "values": st["cache"].values}


_PREPARE = {"tiny": _tiny_prepare, "layer": _layer_prepare, "attention": _attention_prepare, "lm_head": _lm_head_prepare,
            "pointwise": _pointwise_prepare, "prefill": _prefill_prepare, "decode": _decode_prepare}
_RUN = {"tiny": _tiny_run, "layer": _layer_run, "attention": _attention_run, "lm_head": _lm_head_run,
        "pointwise": _pointwise_run, "prefill": _prefill_run, "decode": _decode_run}


# ------------------------------------------------------------------------------------------ work and tolerance
def _layer_weights(h, i, hq, hkv, d):
    return h * d * (2 * hq + 2 * hkv) + 3 * h * i


def work(case):
    """Bytes: every input read once and every output written once; flops: 2 per multiply-add of the
    contractions, causal attention at half of the square."""
    kind = case["kind"]
    if kind == "decode":
        b, t, n = case["batch"], case["context"], DECODE_LAYERS
        wl = _layer_weights(H, I, HQ, HKV, D)
        kv = 2 * b * HKV * D * (t + 1)
        return {"bytes": 2 * (n * (wl + kv) + V * H + b * H + b * V),
                "flops": 2 * b * (n * wl + V * H) + 4 * n * b * HQ * D * (t + 1)}
    b, s = case["batch"], case["seq"]
    t = b * s
    if kind == "tiny":
        e = 4 if case["dtype"] == "f32" else 2
        wl = _layer_weights(TH, TI, THQ, THKV, TD)
        return {"bytes": 2 * e * (TL * wl + 2 * TV * TH) + e * t * TV,
                "flops": 6 * t * (TL * wl + TV * TH) + 3.5 * 2 * TL * b * THQ * s * s * TD}
    if kind == "layer":
        wl = _layer_weights(H, I, HQ, HKV, D)
        return {"bytes": 2 * (2 * wl + 4 * t * H), "flops": 6 * t * wl + 3.5 * 2 * b * HQ * s * s * D}
    if kind == "attention":
        return {"bytes": 2 * 4 * t * D * (HQ + HKV), "flops": 3.5 * 2 * b * HQ * s * s * D}
    if kind == "lm_head":
        return {"bytes": 2 * (2 * V * H + 2 * t * H), "flops": 6 * t * V * H}
    if kind == "pointwise":
        # forward: x, q, k, g, u read and n, q, k, y written; backward: those inputs and the upstream
        # gradients read, the input gradients written
        nqk = HQ * D + HKV * D
        return {"bytes": 2 * t * (5 * (H + nqk) + 8 * I), "flops": 0}
    n = PREFILL_LAYERS
    wl = _layer_weights(H, I, HQ, HKV, D)
    return {"bytes": 2 * (n * (wl + 2 * t * HKV * D) + V * H + t * H + b * V),
            "flops": 2 * (t * n * wl + b * V * H) + 2 * n * b * HQ * s * s * D}


def tolerance(case):
    """About four times the error against 64 bits that one rounding per operator leaves (measured: attention
    2.5e-3 in bf16 and 3e-4 in fp16, LM head and bandwidth-bound operators 1.8e-3, a decoder layer's
    gradients 9e-3, logits after two to four layers and the tiny model's gradients 1.4e-2)."""
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.25e-3}
    if kind in ("pointwise", "lm_head"):
        return {"rel": 7e-3}
    if kind == "tiny" and case["dtype"] == "f32":
        return {"rel": 2e-5}
    return {"rel": 3e-2}


# ------------------------------------------------------------------------------------------ 64-bit results
def _f64(t):
    return t.detach().double()


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope64(x, cos, sin):
    """x [B,S,heads,D]; cos / sin [B,S,D]."""
    h = x.shape[-1] // 2
    return x * cos[:, :, None] + torch.cat((-x[..., h:], x[..., :h]), -1) * sin[:, :, None]


def _attention64(q, k, v):
    """Causal grouped attention of [B,S,heads,D] q against [B,T,heads,D] k / v (q is the suffix), one
    key/value head at a time."""
    b, s, hq, d = q.shape
    t, hk = k.shape[1], k.shape[2]
    mask = torch.ones(s, t, dtype=torch.bool, device=q.device).triu(t - s + 1)
    rows = []
    for bi in range(b):
        heads = []
        for hi in range(hk):
            qi = q[bi, :, hi * (hq // hk):(hi + 1) * (hq // hk)].transpose(0, 1).contiguous()   # [group, S, D]
            p = (qi @ k[bi, :, hi].t().contiguous() * d ** -0.5).masked_fill(mask, -math.inf).softmax(-1)
            heads.append(p @ v[bi, :, hi].contiguous())
        rows.append(torch.cat(heads, 0).transpose(0, 1))
    return torch.stack(rows)


def _mlp64(x, wg, wu, wd):
    return F.linear(F.silu(F.linear(x, wg)) * F.linear(x, wu), wd)


def _layer64(x, p, prefix, cos, sin, d, past=None):
    """A decoder layer in 64 bits; ``p`` maps parameter names to 64-bit tensors.  Returns the output and
    this call's keys and values [B,S,heads,D]."""
    b, s, _ = x.shape
    w = lambda n: p[prefix + n + ".weight"]  # noqa: E731
    h = _norm64(x, w("input_layernorm"))
    q, k, v = (F.linear(h, w(f"self_attn.{n}_proj")).view(b, s, -1, d) for n in "qkv")
    q = _rope64(_norm64(q, w("self_attn.q_norm")), cos, sin)
    k = _rope64(_norm64(k, w("self_attn.k_norm")), cos, sin)
    ka, va = (k, v) if past is None else (torch.cat((past[0], k), 1), torch.cat((past[1], v), 1))
    x = x + F.linear(_attention64(q, ka, va).reshape(b, s, -1), w("self_attn.o_proj"))
    h = _norm64(x, w("post_attention_layernorm"))
    return x + _mlp64(h, w("mlp.gate_proj"), w("mlp.up_proj"), w("mlp.down_proj")), ka, va


def _tables64(positions, d):
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d))
    a = positions.double()[..., None] * inv
    a = torch.cat((a, a), -1)
    return a.cos(), a.sin()


def _mean_ce64(logits, labels):
    return F.cross_entropy(logits[:, :-1].reshape(-1, logits.shape[-1]), labels[:, 1:].reshape(-1), ignore_index=-100)


def _tiny_exact(case, st):
    m, ids = st["model"], st["ids"]
    p = {n: _f64(t).requires_grad_() for n, t in sorted(m.named_parameters())}
    x = F.embedding(ids, p["model.embed_tokens.weight"])
    cos, sin = _tables64(torch.arange(ids.shape[1], device="cuda").expand(ids.shape), TD)
    for i in range(TL):
        x = _layer64(x, p, f"model.layers.{i}.", cos, sin, TD)[0]
    logits = F.linear(_norm64(x, p["model.norm.weight"]), p["lm_head.weight"])
    loss = _mean_ce64(logits, ids)
    return {"logits": logits, "loss": loss, "grads": list(torch.autograd.grad(loss, list(p.values())))}


def _layer_exact(case, st):
    p = {n: _f64(t).requires_grad_() for n, t in sorted(st["layer"].named_parameters())}
    x = _f64(st["x"]).requires_grad_()
    cos, sin = (_f64(t) for t in st["tables"])
    y = _layer64(x, p, "", cos, sin, D)[0]
    return {"y": y, "grads": list(torch.autograd.grad(y, [x, *p.values()], _f64(st["dy"])))}


def _attention_exact(case, st):
    # one batch row and key/value head at a time, each with its own backward: the scores of 8192 positions
    # for every head at once would not fit beside their gradients
    (q, k, v), do = (list(map(_f64, st["qkv"])), _f64(st["do"]))
    g = HQ // HKV
    o, dq, dk, dv = (torch.empty_like(t) for t in (q, q, k, v))
    for bi in range(case["batch"]):
        for hi in range(HKV):
            qs = (slice(bi, bi + 1), slice(None), slice(hi * g, (hi + 1) * g))
            ks = (slice(bi, bi + 1), slice(None), slice(hi, hi + 1))
            leaf = [t.clone().requires_grad_() for t in (q[qs], k[ks], v[ks])]
            oo = _attention64(*leaf)
            o[qs] = oo.detach()
            dq[qs], dk[ks], dv[ks] = torch.autograd.grad(oo, leaf, do[qs])
    return {"o": o, "grads": [dq, dk, dv]}


def _lm_head_exact(case, st):
    x, lab = _f64(st["x"]).view(-1, H), st["labels"]
    b, s = lab.shape
    tgt = torch.full_like(lab, -100)
    tgt[:, :-1] = lab[:, 1:]
    tgt = tgt.view(-1)
    valid = tgt != -100
    n = valid.sum()
    chunk = 8192
    lse = torch.full((b * s,), -math.inf, device="cuda", dtype=torch.float64)
    pick = torch.zeros_like(lse)
    for c in range(0, V, chunk):
        z = x @ _f64(st["w"][c:c + chunk]).t()
        lse = torch.logaddexp(lse, z.logsumexp(-1))
        own = valid & (tgt >= c) & (tgt < c + z.shape[1])
        pick[own] = z[own, tgt[own] - c]
    loss = ((lse - pick) * valid).sum() / n
    dx, dw = torch.zeros_like(x), torch.empty(V, H, device="cuda", dtype=torch.float64)
    for c in range(0, V, chunk):
        w = _f64(st["w"][c:c + chunk])
        z = ((x @ w.t()) - lse[:, None]).exp_()
        own = valid & (tgt >= c) & (tgt < c + z.shape[1])
        z[own, tgt[own] - c] -= 1
        z *= (valid / n)[:, None]
        dx += z @ w
        dw[c:c + chunk] = z.t() @ x
    return {"loss": loss, "dx": dx.view(b, s, H), "dw": dw}


def _pointwise_exact(case, st):
    t = {n: _f64(x).requires_grad_() for n, x in st["t"].items()}
    w = {n: _f64(x).requires_grad_() for n, x in st["w"].items()}
    up = {n: _f64(x) for n, x in st["up"].items()}
    cos, sin = (_f64(x) for x in st["tables"])
    n = _norm64(t["x"], w["x"])
    q, k = (_rope64(_norm64(t[i], w[i]), cos, sin) for i in "qk")
    y = F.silu(t["g"]) * t["u"]
    dx = torch.autograd.grad(n, [t["x"], w["x"]], up["x"])
    dqk = torch.autograd.grad([q, k], [t["q"], t["k"], w["q"], w["k"]], [up["q"], up["k"]])
    dgu = torch.autograd.grad(y, [t["g"], t["u"]], up["g"])
    return {"out": [n, q, k, y], "grads": [*dx, *dqk, *dgu]}


@torch.no_grad()
def _serve_exact(case, st, layers):
    m, ids = st["model"], st["ids"]
    named = dict(m.named_parameters())
    start = st.get("context", 0)
    x = _f64(named["model.embed_tokens.weight"][ids])
    cos, sin = _tables64(torch.arange(start, start + ids.shape[1], device="cuda").expand(ids.shape), D)
    keys, values = [], []
    for i in range(layers):
        pre = f"model.layers.{i}."
        p = {n: _f64(t) for n, t in named.items() if n.startswith(pre)}
        past = None if start == 0 else tuple(_f64(c[i][:, :, :start]).transpose(1, 2)
                                             for c in (st["cache"].keys, st["cache"].values))
        x, k, v = _layer64(x, p, pre, cos, sin, D, past)
        keys.append(k.transpose(1, 2).contiguous())
        values.append(v.transpose(1, 2).contiguous())
    x = _norm64(x[:, -1:], _f64(named["model.norm.weight"]))
    return {"logits": F.linear(x, _f64(named["lm_head.weight"])), "keys": keys, "values": values}


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "prefill":
        return _serve_exact(case, st, PREFILL_LAYERS)
    if kind == "decode":
        return _serve_exact(case, st, DECODE_LAYERS)
    return {"tiny": _tiny_exact, "layer": _layer_exact, "attention": _attention_exact, "lm_head": _lm_head_exact,
            "pointwise": _pointwise_exact}[kind](case, st)
