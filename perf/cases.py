"""Timed workloads of the library: what a program that decodes or prefills with it calls.

Sizes are the ones this repository's benchmark and tests use (16 heads x 128, hidden
2048, FFN 5504, vocabulary 151936, 24 layers; KV lengths 512 to 32768; prompts of 100 to
2048 tokens); `draw` spreads heads, hidden sizes, lengths, layouts and options over the
range the entry points accept.  Inputs are synthetic: activations N(0, 1), weights
N(0, 0.02^2) as the library's own random models, K rows N(0, 0.5^2).

Calls that a decode step makes once per layer are made over several layers with their own
weights and caches, as the step makes them, so that no layer finds its operands in a cache
that the layer itself filled.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-inference-diy_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qdiy  # noqa: E402

D = qdiy.HEAD_DIM
EPS = 1e-6
ROPE_BASE = 10000.0
DEV = "cuda"


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one attention call over a short context: the smallest call, launch and host cost
        dict(name="attn_512", kind="attn", heads=16, rows=512, layers=1, spikes=False, layout="engine"),
        # split-KV attention over a long context, the benchmark's headline length, layer by layer
        dict(name="attn_8192", kind="attn", heads=16, rows=8192, layers=4, spikes=False, layout="engine"),
        # the longest context, 1% of the keys scaled up (the merge then sees large score spreads)
        dict(name="attn_32768_spikes", kind="attn", heads=16, rows=32768, layers=2, spikes=True,
             layout="engine"),
        # a decode step's attention section: RMSNorm + QKV + bias + RoPE + append + attention
        dict(name="front_attn_2048", kind="front", heads=16, pos=2047, layers=12, norm=True, bias=True),
        # the rest of a decode step's layers: output projection, SwiGLU FFN, down projection
        dict(name="decode_mlp_5504", kind="mlp", hidden=2048, inter=5504, layers=8),
        # a layer's projections over a chat-sized prompt in the default (exact) mode
        dict(name="exact_proj_127", kind="proj", mode="exact", tokens=127, hidden=2048, inter=5504, layers=1),
        # the same over a ragged chunk of a long prompt
        dict(name="exact_proj_1000", kind="proj", mode="exact", tokens=1000, hidden=2048, inter=5504, layers=1),
        # a layer's projections on the matrix cores: short prompt, weights not yet in a cache
        dict(name="mfma_proj_100", kind="proj", mode="mfma", tokens=100, hidden=2048, inter=5504, layers=3),
        # and over a full 2048-token pass
        dict(name="mfma_proj_2048", kind="proj", mode="mfma", tokens=2048, hidden=2048, inter=5504, layers=1),
        # causal prompt attention, default mode: a chunk in the middle of a long prompt
        dict(name="exact_attn_256_at_768", kind="prefill", mode="exact", heads=16, tokens=256, pos0=768),
        # causal prompt attention on the matrix cores over a full pass
        dict(name="mfma_attn_2048", kind="prefill", mode="mfma", heads=16, tokens=2048, pos0=0),
        # the engine, whole: a 128-token prompt in the default mode, then decode steps
        dict(name="engine_128_32", kind="engine", mode="exact", layers=24, heads=16, inter=5504, vocab=151936,
             prompt=128, steps=32),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(("attn", "attn", "front", "mlp", "proj", "proj", "prefill", "prefill", "engine"))
    if kind == "attn":
        heads = rng.choice((4, 8, 12, 16, 16, 20, 24, 32))
        rows = _log_int(rng, 1, 32768)
        layers = max(1, min(4, 65536 * 16 // (rows * heads)))
        return dict(kind=kind, heads=heads, rows=rows, layers=rng.randint(1, layers), spikes=rng.random() < 0.3,
                    layout=rng.choice(("engine", "engine", "head_major", "padded")))
    if kind == "front":
        return dict(kind=kind, heads=rng.choice((4, 8, 8, 12, 16, 16, 20, 24, 32)), pos=_log_int(rng, 1, 4096) - 1,
                    layers=rng.randint(1, 6), norm=rng.random() < 0.8, bias=rng.random() < 0.8)
    if kind == "mlp":
        hidden = 512 * rng.randint(1, 8)
        return dict(kind=kind, hidden=hidden, inter=8 * _log_int(rng, 40, 1024), layers=rng.randint(1, 4))
    if kind == "proj":
        mode = rng.choice(("exact", "mfma"))
        tokens = _log_int(rng, 1, 1000 if mode == "exact" else 2048)
        return dict(kind=kind, mode=mode, tokens=tokens, hidden=512 * rng.randint(1, 4),
                    inter=64 * rng.randint(8, 86) if mode == "mfma" else 8 * rng.randint(64, 688), layers=1)
    if kind == "prefill":
        mode = rng.choice(("exact", "mfma"))
        tokens = _log_int(rng, 1, 256 if mode == "exact" else 2048)
        pos0 = rng.choice((0, _log_int(rng, 1, 2048)))
        return dict(kind=kind, mode=mode, heads=rng.choice((4, 8, 12, 16, 16)), tokens=tokens,
                    pos0=min(pos0, 1024 if mode == "exact" else 2048))
    return dict(kind="engine", mode=rng.choice(("exact", "exact", "mfma")), layers=rng.randint(1, 4),
                heads=rng.choice((4, 8, 12, 16)), inter=64 * rng.randint(8, 86), vocab=rng.randint(1000, 40000),
                prompt=_log_int(rng, 1, 512), steps=rng.randint(1, 16))


# ------------------------------------------------------------------- the inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0, mean=0.0):
    t = torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, 1.0, generator=g)
    return t.mul_(scale).add_(mean).half()


def _strides(case):
    """(row stride, head stride, elements) of one cache of case["rows"] rows."""
    heads, rows = case["heads"], case["rows"]
    if case["layout"] == "head_major":
        return D, rows * D, heads * rows * D
    row = heads * D + (64 if case["layout"] == "padded" else 0)
    return row, D, rows * row


def _attn_inputs(case, seed):
    g = _gen(seed)
    rs, hs, n = _strides(case)
    layers = []
    for _ in range(case["layers"]):
        q = _randn(g, case["heads"], D)
        k = _randn(g, n, scale=0.5)
        v = _randn(g, n)
        if case["spikes"]:
            view = k.as_strided((case["rows"], case["heads"], D), (rs, hs, 1))
            hit = torch.rand((case["rows"], case["heads"], 1), device=DEV, generator=g) < 0.01
            view.mul_(torch.where(hit, 8.0, 1.0).half())
        layers.append((q, k, v))
    return layers


def _front_inputs(case, seed):
    g = _gen(seed)
    hid = case["heads"] * D
    layers = []
    for _ in range(case["layers"]):
        x = _randn(g, hid)
        norm = _randn(g, hid, scale=0.1, mean=1.0) if case["norm"] else None
        w = _randn(g, 3 * hid, hid, scale=0.02)
        bias = _randn(g, 3 * hid, scale=0.02) if case["bias"] else None
        k = _randn(g, case["pos"] + 1, hid, scale=0.5)
        v = _randn(g, case["pos"] + 1, hid)
        layers.append((x, norm, w, bias, k, v))
    return layers


def _mlp_inputs(case, seed):
    g = _gen(seed)
    hid, inter = case["hidden"], case["inter"]
    x = _randn(g, hid)
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(att=_randn(g, hid), wo=_randn(g, hid, hid, scale=0.02),
                           norm=_randn(g, hid, scale=0.1, mean=1.0), w1=_randn(g, inter, hid, scale=0.02),
                           w2=_randn(g, inter, hid, scale=0.02), wd=_randn(g, hid, inter, scale=0.02)))
    return x, layers


def _proj_inputs(case, seed):
    g = _gen(seed)
    m, hid, inter = case["tokens"], case["hidden"], case["inter"]
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(x=_randn(g, m, hid), att=_randn(g, m, hid), res=_randn(g, m, hid),
                           act=_randn(g, m, inter, scale=0.5), wqkv=_randn(g, 3 * hid, hid, scale=0.02),
                           wo=_randn(g, hid, hid, scale=0.02), w1=_randn(g, inter, hid, scale=0.02),
                           w2=_randn(g, inter, hid, scale=0.02), wd=_randn(g, hid, inter, scale=0.02)))
    return layers


def _prefill_inputs(case, seed):
    g = _gen(seed)
    hid, rows = case["heads"] * D, case["pos0"] + case["tokens"]
    return _randn(g, case["tokens"], 3 * hid), _randn(g, rows, hid, scale=0.5), _randn(g, rows, hid)


def _engine_cfg(case):
    return qdiy.model_cfg(vocab_size=case["vocab"], hidden_size=case["heads"] * D, num_layers=case["layers"],
                          num_heads=case["heads"], intermediate_size=case["inter"], max_seqlen=2048)


def _engine_tokens(case, seed):
    rng = np.random.default_rng(seed)
    return [int(t) for t in rng.integers(0, case["vocab"], case["prompt"] - 1 + case["steps"])]


def _engine_image(case, seed):
    threads = max(1, min(16, len(os.sched_getaffinity(0))))
    return qdiy.random_model_image(_engine_cfg(case), seed, 0.02, threads)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "attn":
        rs, hs, _ = _strides(case)
        st["ctx"] = qdiy.Context(num_heads=case["heads"], max_seqlen=case["rows"], kv_row_stride=rs,
                                 kv_head_stride=hs)
        st["layers"] = [(q, k, v, torch.empty_like(q)) for q, k, v in _attn_inputs(case, seed)]
    elif kind == "front":
        hid = case["heads"] * D
        st["ctx"] = qdiy.Context(num_heads=case["heads"], max_seqlen=case["pos"] + 1)
        st["layers"] = [(*t, torch.empty(3 * hid, dtype=torch.float16, device=DEV),
                         torch.empty(hid, dtype=torch.float16, device=DEV)) for t in _front_inputs(case, seed)]
    elif kind == "mlp":
        x, layers = _mlp_inputs(case, seed)
        for p in layers:
            p["mid"], p["out"] = torch.empty_like(x), torch.empty_like(x)
            p["act"] = torch.empty(case["inter"], dtype=torch.float16, device=DEV)
        st["x"], st["layers"] = x, layers
    elif kind == "proj":
        m, hid, inter = case["tokens"], case["hidden"], case["inter"]
        st["layers"] = _proj_inputs(case, seed)
        new = lambda n: torch.empty((m, n), dtype=torch.float16, device=DEV)
        for p in st["layers"]:
            p["y_qkv"], p["y_o"], p["y_d"] = new(3 * hid), new(hid), new(hid)
            p["y_ff"] = [new(inter)] if case["mode"] == "mfma" else [new(inter), new(inter)]
    elif kind == "prefill":
        qkv, k, v = _prefill_inputs(case, seed)
        st["ctx"] = qdiy.Context(num_heads=case["heads"], max_seqlen=k.shape[0])
        st.update(qkv=qkv, k=k, v=v, out=torch.empty((case["tokens"], case["heads"] * D), dtype=torch.float16,
                                                     device=DEV))
    else:
        st["eng"] = qdiy.Engine(image=_engine_image(case, seed))
        st["eng"].set_prefill_mode(qdiy.GEMM_MFMA if case["mode"] == "mfma" else qdiy.GEMM_EXACT)
        st["tokens"] = _engine_tokens(case, seed)
    return st


# --------------------------------------------------------------------- one pass

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "attn":
        ctx, rows = st["ctx"], case["rows"]
        return [ctx.decode_attention(q, k, v, out, rows) for q, k, v, out in st["layers"]]
    if kind == "front":
        ctx, pos = st["ctx"], case["pos"]
        res = []
        for x, norm, w, bias, k, v, qkv, out in st["layers"]:
            ctx.qkv_proj_rope_cache_attention(x, norm, w, bias, qkv, k, v, out, pos, EPS)
            res.append([qkv, k, v, out])
        return res
    if kind == "mlp":
        hid, inter = case["hidden"], case["inter"]
        x, res = st["x"], []
        for p in st["layers"]:
            qdiy.proj_residual(p["att"], p["wo"], x, p["mid"], hid, hid)
            qdiy.ffn_up_swiglu(p["mid"], p["norm"], p["w1"], p["w2"], p["act"], hid, inter, EPS)
            x = qdiy.proj_residual(p["act"], p["wd"], p["mid"], p["out"], hid, inter)
            res.append([p["mid"], p["act"], x])
        return res
    if kind == "proj":
        m, hid, inter = case["tokens"], case["hidden"], case["inter"]
        mode = qdiy.GEMM_MFMA if case["mode"] == "mfma" else qdiy.GEMM_EXACT
        res = []
        for p in st["layers"]:
            qdiy.gemm_nt(p["x"], p["wqkv"], p["y_qkv"], m, 3 * hid, hid, mode=mode)
            qdiy.gemm_nt(p["att"], p["wo"], p["y_o"], m, hid, hid, residual=p["res"], mode=mode)
            if mode == qdiy.GEMM_MFMA:
                qdiy.gemm_swiglu(p["x"], p["w1"], p["w2"], p["y_ff"][0], m, inter, hid)
            else:
                qdiy.gemm_nt(p["x"], p["w1"], p["y_ff"][0], m, inter, hid)
                qdiy.gemm_nt(p["x"], p["w2"], p["y_ff"][1], m, inter, hid)
            qdiy.gemm_nt(p["act"], p["wd"], p["y_d"], m, hid, inter, residual=p["res"], mode=mode)
            res.append([p["y_qkv"], p["y_o"], *p["y_ff"], p["y_d"]])
        return res
    if kind == "prefill":
        mode = qdiy.GEMM_MFMA if case["mode"] == "mfma" else qdiy.GEMM_EXACT
        return st["ctx"].prefill_attention(st["qkv"], st["k"], st["v"], st["out"], case["pos0"], case["tokens"],
                                           mode, q_stride=3 * case["heads"] * D)
    eng, toks, n = st["eng"], st["tokens"], case["prompt"] - 1
    pos = eng.prefill(toks[:n]) if n else 0
    nxt = [eng.step(t, pos + i) for i, t in enumerate(toks[n:])]
    k, v = eng.kv_rows(case["layers"] - 1, 0, n + case["steps"])
    return dict(next=np.array(nxt, np.int64), logits=eng.logits(), k=k, v=v)


# ------------------------------------------------------------ what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "attn":
        per = case["heads"] * D * case["rows"]
        return dict(bytes=case["layers"] * (4 * per + 4 * case["heads"] * D), flops=case["layers"] * 4 * per)
    if kind == "front":
        hid, rows = case["heads"] * D, case["pos"] + 1
        return dict(bytes=case["layers"] * (6 * hid * hid + 4 * hid * rows + 2 * 12 * hid),
                    flops=case["layers"] * (6 * hid * hid + 4 * hid * rows))
    if kind == "mlp":
        n = case["hidden"] * (case["hidden"] + 3 * case["inter"])
        return dict(bytes=case["layers"] * (2 * n + 2 * (6 * case["hidden"] + case["inter"])),
                    flops=case["layers"] * 2 * n)
    if kind == "proj":
        m, hid, inter = case["tokens"], case["hidden"], case["inter"]
        n = hid * (4 * hid + 3 * inter)
        outs = 1 if case["mode"] == "mfma" else 2
        return dict(bytes=case["layers"] * 2 * (n + m * (8 * hid + inter * (1 + outs))),
                    flops=case["layers"] * 2 * n * m)
    if kind == "prefill":
        hid, t, p = case["heads"] * D, case["tokens"], case["pos0"]
        return dict(bytes=2 * hid * (2 * (p + t) + 2 * t), flops=4 * hid * (t * p + t * (t + 1) // 2))
    hid, inter, layers = case["heads"] * D, case["inter"], case["layers"]
    n, s, vocab = case["prompt"] - 1, case["steps"], case["vocab"]
    per_layer = hid * (4 * hid + 3 * inter)
    rows = [n + i + 1 for i in range(s)]
    weights = 2 * layers * per_layer
    return dict(bytes=(weights if n else 0) + s * (weights + 2 * vocab * hid) + layers * 4 * hid * (sum(rows) + n),
                flops=2 * layers * per_layer * (n + s) + 2 * vocab * hid * s
                + layers * 4 * hid * (sum(rows) + n * (n + 1) // 2))


# --------------------------------------------------------------- how far apart is right

def tolerance(case):
    """About four times the distance measured between the library and `exact`, which is the
    rounding of fp16 outputs (2e-4) and, where a chain stores fp16 in between, of those."""
    kind = case["kind"]
    if kind == "attn":
        return dict(rel=8e-4)                  # measured 2.1e-4
    if kind == "front":
        return dict(rel=1.6e-3)                # 3.8e-4
    if kind == "mlp":
        return dict(rel=4e-3)                  # 1e-3 after four layers
    if kind == "proj":
        return dict(rel=1.6e-3)                # 3.9e-4 (the SwiGLU)
    if kind == "prefill":
        return dict(rel=8e-4 if case["mode"] == "exact" else 1.2e-3)   # 2.1e-4 and 2.7e-4
    return dict(rel=1.6e-2, differ=0.2)        # 3.9e-3 over 24 layers; tokens: near-ties of random logits


# ------------------------------------------------------------------ the same in 64 bits

def _attend(q, k, v):
    """Softmax attention of one query per head, float64: q [H, D], k and v [rows, H, D]."""
    s = torch.einsum("hd,lhd->hl", q, k) / math.sqrt(D)
    return torch.einsum("hl,lhd->hd", torch.softmax(s, dim=1), v)


def _causal(q, k, v, pos0):
    """Causal attention, float64: q [T, H, D] at positions pos0.., k and v [pos0 + T, H, D]."""
    t, heads = q.shape[0], q.shape[1]
    out = torch.empty_like(q)
    keep = torch.arange(k.shape[0], device=q.device)[None, :] <= pos0 + torch.arange(t, device=q.device)[:, None]
    for h in range(heads):
        s = (q[:, h] @ k[:, h].t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(~keep, -math.inf), dim=1) @ v[:, h].contiguous()
    return out


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w


def _rope(x, pos):
    """Rotate-half RoPE, float64: x [T, H, D] at integer positions pos [T]."""
    inv = ROPE_BASE ** (-torch.arange(0, D, 2, dtype=torch.float64, device=x.device) / D)
    ang = pos.double()[:, None] * inv[None, :]
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _swiglu(g, u):
    return g * (u / (1.0 + torch.exp(-u)))


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        rs, hs, _ = _strides(case)
        shape, stride = (case["rows"], case["heads"], D), (rs, hs, 1)
        return [_attend(q.double(), k.as_strided(shape, stride).double(), v.as_strided(shape, stride).double())
                for q, k, v in _attn_inputs(case, seed)]
    if kind == "front":
        heads, hid, pos = case["heads"], case["heads"] * D, case["pos"]
        at = torch.tensor([pos], device=DEV)
        res = []
        for x, norm, w, bias, k, v in _front_inputs(case, seed):
            xn = x.double() if norm is None else _rms(x.double(), norm.double())
            qkv = w.double() @ xn
            if bias is not None:
                qkv = qkv + bias.double()
            q = _rope(qkv[:hid].view(1, heads, D), at)[0]
            k, v = k.double(), v.double()
            k[pos] = _rope(qkv[hid:2 * hid].view(1, heads, D), at).view(hid)
            v[pos] = qkv[2 * hid:]
            out = _attend(q, k.view(-1, heads, D), v.view(-1, heads, D))
            res.append([torch.cat((q.reshape(hid), qkv[hid:])), k, v, out.reshape(hid)])
        return res
    if kind == "mlp":
        x, layers = _mlp_inputs(case, seed)
        x, res = x.double(), []
        for p in layers:
            p = {n: t.double() for n, t in p.items()}
            mid = x + p["wo"] @ p["att"]
            xn = _rms(mid, p["norm"])
            act = _swiglu(p["w1"] @ xn, p["w2"] @ xn)
            x = mid + p["wd"] @ act
            res.append([mid, act, x])
        return res
    if kind == "proj":
        res = []
        for p in _proj_inputs(case, seed):
            p = {n: t.double() for n, t in p.items()}
            g, u = p["x"] @ p["w1"].t(), p["x"] @ p["w2"].t()
            ff = [_swiglu(g, u)] if case["mode"] == "mfma" else [g, u]
            res.append([p["x"] @ p["wqkv"].t(), p["res"] + p["att"] @ p["wo"].t(), *ff,
                        p["res"] + p["act"] @ p["wd"].t()])
        return res
    if kind == "prefill":
        qkv, k, v = _prefill_inputs(case, seed)
        t, heads = case["tokens"], case["heads"]
        q = qkv[:, :heads * D].double().view(t, heads, D)
        return _causal(q, k.double().view(-1, heads, D), v.double().view(-1, heads, D), case["pos0"]).view(t, -1)
    return _engine_exact(case, seed)


def _engine_exact(case, seed):
    """The whole model in float64 over prompt and steps at once (the steps' tokens are given)."""
    heads, hid, inter, vocab = case["heads"], case["heads"] * D, case["inter"], case["vocab"]
    img = _engine_image(case, seed)[28:].view(np.float16)
    toks = torch.tensor(_engine_tokens(case, seed))
    at = 0

    def take(*shape):
        nonlocal at
        n = math.prod(shape)
        t = torch.from_numpy(img[at:at + n])
        at += n
        return t.view(*shape)

    dev = lambda t: t.to(DEV).double()
    n = toks.numel()
    pos = torch.arange(n, device=DEV)
    x = dev(take(vocab, hid)[toks])
    for _ in range(case["layers"]):
        ln_1, wqkv, bqkv = dev(take(hid)), dev(take(3 * hid, hid)), dev(take(3 * hid))
        wo, ln_2 = dev(take(hid, hid)), dev(take(hid))
        w1, w2, wd = dev(take(inter, hid)), dev(take(inter, hid)), dev(take(hid, inter))
        qkv = (_rms(x, ln_1) @ wqkv.t() + bqkv).view(n, 3, heads, D)
        q, k, v = _rope(qkv[:, 0], pos), _rope(qkv[:, 1], pos), qkv[:, 2]
        x = x + _causal(q, k, v, 0).view(n, hid) @ wo.t()
        xn = _rms(x, ln_2)
        x = x + _swiglu(xn @ w1.t(), xn @ w2.t()) @ wd.t()
    ln_f, head = dev(take(hid)), take(vocab, hid)
    xn = _rms(x[-1], ln_f)
    logits = torch.cat([dev(head[i:i + 16384]) @ xn for i in range(0, vocab, 16384)])
    host = lambda t: t.reshape(-1, hid).cpu().numpy() if t.dim() > 1 else t.cpu().numpy()
    return dict(next=None, logits=host(logits), k=host(k), v=host(v))
