"""The work a user of this framework has it do, as measurable cases.

``listed()`` names twelve of them, from one short prompt's attention to a whole cached GPT-2
generation; ``draw()`` makes more of the same ranges.  Each goes through the public entry points
(custom_flash_attn.forward / forward_lse / attention / flash_attn_forward / decode, and the GPT-2
modules of model_inference) the way a program calls them.  Sizes are those of the GPT-2 family
(12 to 25 heads of 64, contexts up to 1024), of the benchmark's long-sequence and head-dim-128
legs, and generic odd ones.

Case fields: ``kind`` picks the entry point ("forward", "attention", "flash", "decode", "layer",
"block", "generate"); the others are its sizes and options.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [os.path.join(_ROOT, "tfg-flashattention_amd")]

import custom_flash_attn as fa  # noqa: E402
import model_inference as mi  # noqa: E402

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MODELS = ("gpt2-small (124M)", "gpt2-medium (355M)", "gpt2-large (774M)", "gpt2-xl (1558M)")


def listed():
    return [
        # One short prompt through GPT-2 small's heads: the smallest call, launch and latency.
        dict(name="forward_prompt", kind="forward", B=1, H=12, N=256, sigma=1.0, lse=False),
        # A batch of full contexts at GPT-2 XL's heads, peaked scores: the benchmark's headline.
        dict(name="forward_batch", kind="forward", B=8, H=25, N=1024, sigma=3.0, lse=False),
        # One long sequence, with the log-sum-exp for a later merge.
        dict(name="forward_long", kind="forward", B=1, H=16, N=8192, sigma=1.0, lse=True),
        # Two ragged prompts of GPT-2 medium: the (B, N, H, d) projections read in place, the
        # context written in the layout the output projection takes.
        dict(name="attention_views_ragged", kind="attention", B=2, H=16, Nq=777, Nk=777, D=64, dtype="bf16",
             causal=True, lse=False, views=True),
        # Unmasked attention of one sequence over another, fp16, a head dim between the compiled
        # ones, with the log-sum-exp.
        dict(name="attention_cross_d80", kind="attention", B=2, H=16, Nq=1000, Nk=1333, D=80, dtype="fp16",
             causal=False, lse=True, views=False),
        # The Triton wrapper's call, fp16, the largest head dim.
        dict(name="flash_fp16_d128", kind="flash", B=8, H=16, Nq=1024, Nk=1024, D=128, dtype="fp16"),
        # One token of one GPT-2 small sequence over a partly filled cache, appended in place.
        dict(name="decode_single", kind="decode", B=1, H=12, N=1024, D=64, dtype="bf16", append=True, lse=False),
        # One token of each of eight GPT-2 XL sequences of unequal lengths.
        dict(name="decode_batch", kind="decode", B=8, H=25, N=1024, D=64, dtype="bf16", append=True, lse=False),
        # Long fp16 caches at head dim 128, no append, with the log-sum-exp.
        dict(name="decode_long_d128", kind="decode", B=4, H=16, N=8192, D=128, dtype="fp16", append=False, lse=True),
        # GPT-2 medium's attention module over a batch of full contexts, under bf16 autocast.
        dict(name="layer_medium", kind="layer", model=MODELS[1], B=4, N=1024),
        # One GPT-2 XL block (attention, norms, MLP, residuals) over a ragged prompt.
        dict(name="block_xl_ragged", kind="block", model=MODELS[3], B=1, N=613),
        # A whole GPT-2 medium generation of a small batch: prompt prefill, then replayed decode
        # steps over given tokens; returns the logits that would be sampled from.
        dict(name="generate_medium", kind="generate", model=MODELS[1], B=4, N=250, steps=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: prompts of 32 to 4096 tokens in batches of 1 to 8 (32 to
    1500 keys unmasked), caches of 128 to 8192 rows, every GPT-2 size for single modules and the
    two smaller ones for whole generations."""
    kind = rng.choice(("forward", "attention", "attention", "flash", "decode", "decode", "layer", "block", "generate"))
    c = dict(kind=kind)
    if kind in ("forward", "attention", "flash"):
        c.update(B=rng.choice((1, 1, 2, 3, 4, 8)), H=rng.choice((12, 16, 20, 25)))
    if kind == "forward":
        c.update(N=_log_int(rng, 32, 4096 if c["B"] <= 2 else 1024), sigma=rng.choice((1.0, 3.0)),
                 lse=rng.random() < 0.5)
    elif kind in ("attention", "flash"):
        c.update(D=rng.choice((64, 64, 128, 128, 32, 40, 72, 80, 96, 120)), dtype=rng.choice(("bf16", "fp16")))
        n = _log_int(rng, 32, 4096 if c["B"] <= 2 else 1024)
        if kind == "flash":
            c.update(Nq=n, Nk=n if rng.random() < 0.5 else _log_int(rng, 32, 2048))
        elif rng.random() < 0.5:
            c.update(Nq=n, Nk=n, causal=True)
        else:
            c.update(Nq=_log_int(rng, 32, 1500), Nk=_log_int(rng, 32, 1500), causal=False)
        if kind == "attention":
            c.update(lse=rng.random() < 0.5, views=rng.random() < 0.5)
    elif kind == "decode":
        B = rng.choice((1, 1, 2, 4, 8, 16))
        c.update(B=B, H=rng.choice((12, 16, 20, 25, 32)), N=_log_int(rng, 128, 8192 if B <= 4 else 2048),
                 D=rng.choice((64, 64, 64, 128, 128, 80)), dtype=rng.choice(("bf16", "fp16")),
                 append=rng.random() < 0.7, lse=rng.random() < 0.3)
    elif kind in ("layer", "block"):
        B = rng.choice((1, 1, 2, 4))
        c.update(model=rng.choice(MODELS), B=B, N=_log_int(rng, 16, 1024))
    else:
        c.update(model=rng.choice(MODELS[:2]), B=rng.choice((1, 1, 2, 3, 4)), N=_log_int(rng, 12, 250),
                 steps=rng.randint(4, 16))
    return c


# ---------------------------------------------------------------------------------------
# Inputs, from the seed alone.


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, shape, dtype, sigma=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * sigma).to(dtype)


def _attention_inputs(case, seed):
    """q, k, v as (B, H, N, D), standard normal (q and k times the forward case's sigma)."""
    g = _gen(seed)
    if case["kind"] == "forward":
        shape = (case["B"], case["H"], case["N"], 64)
        s = case["sigma"]
        return _randn(g, shape, torch.bfloat16, s), _randn(g, shape, torch.bfloat16, s), _randn(g, shape, torch.bfloat16)
    dt = DTYPES[case["dtype"]]
    B, H, D = case["B"], case["H"], case["D"]
    if case.get("views"):
        return tuple(_randn(g, (B, n, H, D), dt).transpose(1, 2) for n in (case["Nq"], case["Nk"], case["Nk"]))
    return tuple(_randn(g, (B, H, n, D), dt) for n in (case["Nq"], case["Nk"], case["Nk"]))


def _decode_lengths(case):
    """Cached rows per sequence: unequal, from half the cache up, one row left for the new token."""
    N = case["N"]
    return [N - 1 - (b * 389 + N // 7) % (N // 2) for b in range(case["B"])]


def _decode_inputs(case, seed):
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    s = dict(q=_randn(g, (B, H, D), dt), k=_randn(g, (B, H, N, D), dt), v=_randn(g, (B, H, N, D), dt),
             kn=_randn(g, (B, H, D), dt), vn=_randn(g, (B, H, D), dt))
    s["lens"] = torch.tensor(_decode_lengths(case), dtype=torch.int32, device=DEV)
    return s


def _cfg(case):
    return mi.gpt2_config(case["model"], impl_type="hip")


def _normal_(module, g):
    """Weights N(0, 0.02^2) as GPT-2 is initialised; biases and norm parameters off their neutral
    values, as a trained checkpoint has them.  Returns name -> tensor."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("scale"):
                p.normal_(1.0, 0.1, generator=g)
            elif name.endswith(("bias", "shift")):
                p.normal_(0.0, 0.05, generator=g)
            else:
                p.normal_(0.0, 0.02, generator=g)
    return dict(module.named_parameters())


def _module(case, seed):
    cfg, g = _cfg(case), _gen(seed)
    with torch.device(DEV):
        if case["kind"] == "layer":
            d = cfg["emb_dim"]
            m = mi.MultiHeadAttention(d, d, cfg["context_length"], 0.0, cfg["n_heads"], "hip", qkv_bias=True)
        elif case["kind"] == "block":
            m = mi.TransformerBlock(cfg)
        else:
            m = mi.GPTModel(cfg)
    m = m.eval()
    return m, _normal_(m, g), g


def _hidden_inputs(case, g):
    return torch.randn((case["B"], case["N"], _cfg(case)["emb_dim"]), generator=g, device=DEV)


def _tokens(case, g):
    return torch.randint(0, _cfg(case)["vocab_size"], (case["B"], case["N"] + case["steps"]), generator=g, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "forward":
        return dict(case=case, qkv=_attention_inputs(case, seed))
    if kind in ("attention", "flash"):
        s = dict(case=case, qkv=_attention_inputs(case, seed))
        if case.get("views"):  # the caller's (B, N, H, d) context buffer
            s["out"] = torch.empty((case["B"], case["Nq"], case["H"], case["D"]), dtype=DTYPES[case["dtype"]], device=DEV)
        return s
    if kind == "decode":
        return dict(case=case, **_decode_inputs(case, seed))
    module, _, g = _module(case, seed)
    if kind == "generate":
        idx = _tokens(case, g)
        return dict(case=case, idx=idx, dec=mi.GraphedDecoder(module, case["B"], case["N"] + case["steps"], DEV))
    return dict(case=case, module=module, x=_hidden_inputs(case, g))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "forward":
        q, k, v = s["qkv"]
        return fa.forward_lse(q, k, v) if case["lse"] else fa.forward(q, k, v)
    if kind == "attention":
        q, k, v = s["qkv"]
        out = s["out"].transpose(1, 2) if case["views"] else None
        return fa.attention(q, k, v, out=out, causal=case["causal"], return_lse=case["lse"])
    if kind == "flash":
        return fa.flash_attn_forward(*s["qkv"])
    if kind == "decode":
        if case["append"]:
            o = fa.decode(s["q"], s["k"], s["v"], s["lens"], s["kn"], s["vn"], return_lse=case["lse"])
            return o, s["k"], s["v"]
        return fa.decode(s["q"], s["k"], s["v"], s["lens"], return_lse=case["lse"])
    if kind == "layer":
        with torch.no_grad(), torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            return s["module"](s["x"])
    if kind == "block":
        with torch.no_grad():
            return s["module"](s["x"])
    # The generation loop of generate_graphed over given tokens, keeping each step's logits.
    dec, idx, n = s["dec"], s["idx"], case["N"]
    dec.cache.reset()
    logits = [dec.prefill(idx[:, :n])]
    for t in range(n, n + case["steps"]):
        logits.append(dec.step(idx[:, t:t + 1]).clone())
    return logits


# ---------------------------------------------------------------------------------------
# What a pass cannot do without.


def _pairs(Nq, Nk, causal):
    if not causal:
        return Nq * Nk
    m = min(Nq, Nk)
    return m * (m + 1) // 2 + max(0, Nq - Nk) * Nk


def _layer_work(cfg, B, N, past=0):
    """flops of one attention module on N new tokens per sequence after `past` cached ones."""
    d = cfg["emb_dim"]
    return 2 * B * N * 4 * d * d + 4 * B * d * (_pairs(N, N, True) + N * past)


def work(case):
    kind = case["kind"]
    if kind in ("forward", "attention", "flash"):
        Nq, Nk, D = case.get("Nq", case.get("N")), case.get("Nk", case.get("N")), case.get("D", 64)
        bh = case["B"] * case["H"]
        nbytes = bh * (4 * Nq * D + 4 * min(Nq if case.get("causal", True) else Nk, Nk) * D + (4 * Nq if case.get("lse") else 0))
        return {"bytes": nbytes, "flops": 4 * bh * D * _pairs(Nq, Nk, case.get("causal", True))}
    if kind == "decode":
        H, D, new = case["H"], case["D"], 1 if case["append"] else 0
        rows = sum(_decode_lengths(case))
        extra = case["B"] * H * (4 * D + new * 8 * D + (4 if case["lse"] else 0))
        return {"bytes": 4 * H * D * rows + extra, "flops": 4 * H * D * (rows + new * case["B"])}
    cfg = _cfg(case)
    d, B, N = cfg["emb_dim"], case["B"], case["N"]
    if kind == "layer":
        return {"bytes": 4 * (4 * d * d + 4 * d) + 6 * B * N * d, "flops": _layer_work(cfg, B, N)}
    block_bytes = 4 * (12 * d * d + 13 * d)
    if kind == "block":
        return {"bytes": block_bytes + 8 * B * N * d, "flops": _layer_work(cfg, B, N) + 16 * B * N * d * d}
    L, V, steps = cfg["n_layers"], cfg["vocab_size"], case["steps"]
    flops = L * (_layer_work(cfg, B, N) + 16 * B * N * d * d) + 2 * B * d * V
    nbytes = L * (block_bytes + 4 * B * N * d) + 4 * V * d + 8 * B * N * d + 4 * B * V
    for t in range(steps):
        flops += L * (_layer_work(cfg, B, 1, N + t) + 16 * B * d * d) + 2 * B * d * V
        nbytes += L * (block_bytes + 4 * B * (N + t + 1) * d) + 4 * V * d + 4 * B * V
    return {"bytes": nbytes, "flops": flops}


# Four times the error against exact() measured over these ranges (rel, max): single attention and
# decode calls 2e-3, 1.7e-2 in bf16 and 2.9e-4, 2.7e-3 in fp16; a module under bf16 autocast 4.5e-3,
# 7.8e-2; a block, whose fp32 residual holds the bf16 attention's error, 1.4e-3, 7.8e-3; a whole
# generation's logits 5.2e-3, 2.4e-2.
_TOLERANCE = {"bf16": (8e-3, 0.07), "fp16": (1.2e-3, 0.011), "layer": (0.018, 0.32), "block": (5.6e-3, 0.032),
              "generate": (0.021, 0.1)}


def tolerance(case):
    rel, largest = _TOLERANCE[case["kind"] if case["kind"] in _TOLERANCE else case.get("dtype", "bf16")]
    return {"rel": rel, "max": largest}


# ---------------------------------------------------------------------------------------
# The same in 64 bits, in plain torch.


def _exact_head(q, k, v, scale, causal):
    """One head in float64, a block of query rows at a time: (o, lse)."""
    Nq, Nk = q.shape[0], k.shape[0]
    kt = k.t().contiguous()
    o = torch.empty((Nq, v.shape[1]), dtype=torch.float64, device=q.device)
    lse = torch.empty(Nq, dtype=torch.float64, device=q.device)
    cols = torch.arange(Nk, device=q.device)
    for i in range(0, Nq, 2048):
        s = (q[i:i + 2048] @ kt) * scale
        if causal:
            s.masked_fill_(cols[None, :] > torch.arange(i, i + s.shape[0], device=q.device)[:, None], -math.inf)
        lse[i:i + 2048] = torch.logsumexp(s, dim=-1)
        o[i:i + 2048] = torch.exp(s - lse[i:i + 2048, None]) @ v
    return o, lse


def _exact_attention(q, k, v, causal):
    B, H, Nq, D = q.shape
    o = torch.empty((B, H, Nq, D), dtype=torch.float64, device=q.device)
    lse = torch.empty((B, H, Nq), dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(H):
            o[b, h], lse[b, h] = _exact_head(q[b, h].double(), k[b, h].double(), v[b, h].double(), 1 / math.sqrt(D), causal)
    return o, lse


def _exact_decode(case, seed):
    s = _decode_inputs(case, seed)
    B, H, D = case["B"], case["H"], case["D"]
    k, v = s["k"].double(), s["v"].double()
    o = torch.empty((B, H, D), dtype=torch.float64, device=DEV)
    lse = torch.empty((B, H), dtype=torch.float64, device=DEV)
    for b, n in enumerate(_decode_lengths(case)):
        if case["append"]:
            k[b, :, n], v[b, :, n] = s["kn"][b].double(), s["vn"][b].double()
            n += 1
        sc = (k[b, :, :n] * s["q"][b, :, None].double()).sum(-1) / math.sqrt(D)
        lse[b] = torch.logsumexp(sc, dim=-1)
        o[b] = (torch.exp(sc - lse[b][:, None])[..., None] * v[b, :, :n]).sum(1)
    r = (o, lse) if case["lse"] else o
    return (r, k, v) if case["append"] else r


def _exact_layer(w, p, x, heads):
    B, N, d = x.shape
    lin = lambda n, t: t @ w[p + n + ".weight"].double().t().contiguous() + w[p + n + ".bias"].double()  # noqa: E731
    q, k, v = (lin(n, x).view(B, N, heads, d // heads).transpose(1, 2) for n in ("W_query", "W_key", "W_value"))
    o, _ = _exact_attention(q, k, v, True)
    return lin("out_proj", o.transpose(1, 2).reshape(B, N, d))


def _exact_norm(w, p, x):
    y = (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, keepdim=True, unbiased=False) + 1e-5)
    return y * w[p + "scale"].double() + w[p + "shift"].double()


def _exact_block(w, p, x, heads):
    x = x + _exact_layer(w, p + "att.", _exact_norm(w, p + "norm1.", x), heads)
    y = _exact_norm(w, p + "norm2.", x)
    y = y @ w[p + "ff.layers.0.weight"].double().t().contiguous() + w[p + "ff.layers.0.bias"].double()
    y = 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3)))
    return x + y @ w[p + "ff.layers.2.weight"].double().t().contiguous() + w[p + "ff.layers.2.bias"].double()


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("forward", "attention", "flash"):
            q, k, v = _attention_inputs(case, seed)
            o, lse = _exact_attention(q, k, v, case.get("causal", True))
            return (o, lse) if case.get("lse") else o
        if kind == "decode":
            return _exact_decode(case, seed)
        _, w, g = _module(case, seed)
        heads = _cfg(case)["n_heads"]
        if kind == "layer":
            return _exact_layer(w, "", _hidden_inputs(case, g).double(), heads)
        if kind == "block":
            return _exact_block(w, "", _hidden_inputs(case, g).double(), heads)
        idx, n = _tokens(case, g), case["N"]
        x = w["tok_emb.weight"].double()[idx] + w["pos_emb.weight"].double()[torch.arange(idx.shape[1], device=DEV)]
        for i in range(_cfg(case)["n_layers"]):
            x = _exact_block(w, "trf_blocks.%d." % i, x, heads)
        x = _exact_norm(w, "final_norm.", x[:, n - 1:])
        head = w["out_head.weight"].double().t().contiguous()
        return [x[:, t] @ head for t in range(case["steps"] + 1)]
