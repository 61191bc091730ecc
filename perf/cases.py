"""Performance cases of the quantized-matmul hot path: what a program that runs a
Q4_K_M decoder on this library spends its time on, each through its public entry
point (the C ABI of include/jllm_hip.h, or the decoder binding).

Sizes are those of the repository's 36-layer decoder configuration (hidden 2560,
32 / 8 heads x 128, ffn 9728, vocabulary 151936, Q4_K with Q6_K downs and head) and
of its tests and benchmark; `draw` spreads over the ranges around them.

A case's "kind":
  gemv          one decode matrix-vector product (gemv_quant, fp16 out)
  head          output norm + vocabulary product of a decode step (fp32 logits)
  decode_step   a greedy decode step of a small stack of full-width layers
  gemm          one prefill product of N tokens (gemm_quant_batched, fp16 out)
  attn_decode   split-K attention of one token over the KV cache
  attn_prefill  causal attention of a prompt chunk over the KV cache
  prompt        the prefill of a prompt through one full-width layer, logits out
"""
import ctypes
import os
import sys

import numpy as np
import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "genie-ai-runtime_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import decoder  # noqa: E402
import jllm  # noqa: E402

DEV = "cuda:0"
Q4, Q5, Q6 = 12, 13, 14
BLOCK = {Q4: 144, Q5: 176, Q6: 210}
HID, QD, FFN, VOCAB = 2560, 4096, 9728, 151936
HEADS, KV, HD = 32, 8, 128
EPS = 1e-6


def listed():
    return [
        # decode: the smallest matrix of a layer (k or v), where latency is all there is
        {"name": "gemv_k", "kind": "gemv", "type": Q4, "M": 1024, "K": HID},
        # decode: the vocabulary product, the largest read of a step
        {"name": "head", "kind": "head", "type": Q6, "M": VOCAB, "K": HID},
        # decode: a whole greedy step in the chat regime (a prompt of some hundred tokens)
        {"name": "decode_step", "kind": "decode_step", "layers": 4, "ctx": 640, "vocab": 16384},
        # prefill of a short question: the widest matrix at a few dozen tokens
        {"name": "gemm_short", "kind": "gemm", "type": Q4, "M": FFN, "K": HID, "N": 33},
        # prefill of a long prompt in one batch, ragged
        {"name": "gemm_prompt", "kind": "gemm", "type": Q4, "M": FFN, "K": HID, "N": 1261},
        # prefill: the Q6_K down projection of a full 512-token chunk
        {"name": "gemm_down", "kind": "gemm", "type": Q6, "M": HID, "K": FFN, "N": 512},
        # prefill of a Q5_K_M model, ragged
        {"name": "gemm_q5k", "kind": "gemm", "type": Q5, "M": FFN, "K": HID, "N": 300},
        # decode attention in the chat regime
        {"name": "attn_decode", "kind": "attn_decode", "heads": HEADS, "kv": KV, "hd": HD, "ctx": 700, "int8": True,
         "window": 0},
        # decode attention over a long document
        {"name": "attn_decode_long", "kind": "attn_decode", "heads": HEADS, "kv": KV, "hd": HD, "ctx": 8192,
         "int8": True, "window": 0},
        # prompt attention: the first chunk of a prompt
        {"name": "attn_prompt", "kind": "attn_prefill", "heads": HEADS, "kv": KV, "hd": HD, "N": 512, "start": 0,
         "int8": True, "window": 0},
        # prompt attention: the last chunk of a long document (chunks of 512 tokens)
        {"name": "attn_prompt_long", "kind": "attn_prefill", "heads": HEADS, "kv": KV, "hd": HD, "N": 512,
         "start": 7680, "int8": True, "window": 0},
        # a layer's whole prefill of a 512-token chunk, with the embedding and the logits
        {"name": "prompt", "kind": "prompt", "layers": 1, "N": 512, "vocab": 4096},
    ]


def _logint(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["gemv", "head", "decode_step", "gemm", "gemm", "gemm", "attn_decode", "attn_decode",
                       "attn_prefill", "attn_prefill", "prompt"])
    if kind == "gemv":
        return {"kind": kind, "type": rng.choice([Q4, Q4, Q5, Q6]), "M": _logint(rng, 256, 2 * FFN),
                "K": 256 * rng.choice([2, 4, 8, 10, 16, 38])}
    if kind == "head":
        return {"kind": kind, "type": rng.choice([Q4, Q6]), "M": _logint(rng, 16000, VOCAB), "K": 256 * rng.choice([8, 10, 16])}
    if kind == "decode_step":
        return {"kind": kind, "layers": rng.choice([2, 3, 4]), "ctx": _logint(rng, 1, 4000),
                "vocab": 256 * rng.randint(8, 64)}
    if kind == "gemm":
        M, K = rng.choice([(1024, HID), (HID, QD), (QD, HID), (FFN, HID), (HID, FFN), (_logint(rng, 200, FFN), HID)])
        return {"kind": kind, "type": rng.choice([Q4, Q4, Q5, Q6]), "M": M, "K": K, "N": _logint(rng, 2, 1261)}
    heads, kv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (16, 4, 128), (8, 2, 64)])
    case = {"kind": kind, "heads": heads, "kv": kv, "hd": hd, "int8": rng.random() < 0.75,
            "window": rng.choice([0, 0, 0, 512])}
    if kind == "attn_decode":
        case["ctx"] = _logint(rng, 1, 8192)
        return case
    if kind == "attn_prefill":
        case["N"] = _logint(rng, 2, 512)
        case["start"] = rng.choice([0, _logint(rng, 1, 7680)])
        return case
    return {"kind": kind, "layers": 1, "N": _logint(rng, 2, 512), "vocab": 4096}


# ---- inputs -----------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _weights(g, t, M, K):
    """Random K-quant rows whose weights have mean about 0 and a standard deviation of
    about 0.02, the block scales of the decoder module's random models."""
    nb = K // 256
    b = torch.randint(0, 256, (M, nb, BLOCK[t]), dtype=torch.uint8, device=DEV, generator=g)
    if t == Q6:
        b[:, :, 192:208] = torch.randint(-32, 32, (M, nb, 16), dtype=torch.int8, device=DEV, generator=g).view(torch.uint8)
        d = torch.randn((M, nb, 1), device=DEV, generator=g).abs() * decoder.Q6_D
        b[:, :, 208:210] = d.half().view(torch.uint8)
    else:
        s = [decoder.Q4_D, decoder.Q4_DMIN] if t == Q4 else [decoder.Q5_D, decoder.Q5_DMIN]
        d = torch.randn((M, nb, 2), device=DEV, generator=g).abs() * torch.tensor(s, device=DEV)
        b[:, :, 0:4] = d.half().view(torch.uint8)
    return b.reshape(-1)


def _kv(g, ctx, kv, hd, int8):
    """K or V rows of a cache: fp16 values, or int8 codes with the scale absmax / 127 of
    each (position, head)."""
    v = torch.randn((ctx, kv, hd), device=DEV, generator=g)
    if not int8:
        return v.half(), None
    sc = v.abs().amax(-1) / 127.0
    return torch.round(v / sc[..., None]).to(torch.int8), sc.contiguous()


def _fn(name, *args):
    """A C-ABI call with its arguments converted once, as a program's binding keeps it."""
    f = getattr(jllm.lib(), name)
    conv = [t(a.data_ptr() if hasattr(a, "data_ptr") else a) if a is not None else None
            for t, a in zip(f.argtypes, args)]
    conv.append(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return f, conv, name


def _tokens(case, seed, n):
    return torch.randint(0, case["vocab"], (n,), dtype=torch.int32, device=DEV, generator=_gen(seed + 77))


def _decoder(case, seed, max_seq):
    shape = decoder.Shape(n_layers=case["layers"], vocab_size=case["vocab"])
    model = decoder.synth_device(shape, int(seed), DEV)
    return shape, model, decoder.Decoder(shape, model, max_seq, max_batch=512)


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("gemv", "head", "gemm"):
        s = {"W": _weights(g, case["type"], case["M"], case["K"]),
             "x": torch.randn((case.get("N", 1), case["K"]), device=DEV, generator=g).half()}
        if kind == "head":
            s["norm"] = 1.0 + 0.02 * torch.randn(case["K"], device=DEV, generator=g)
        return s
    ctx = case["ctx"] if kind == "attn_decode" else case["start"] + case["N"]
    k, ks = _kv(g, ctx, case["kv"], case["hd"], case["int8"])
    v, vs = _kv(g, ctx, case["kv"], case["hd"], case["int8"])
    q = torch.randn((case.get("N", 1), case["heads"], case["hd"]), device=DEV, generator=g).half()
    return {"q": q, "k": k, "v": v, "ks": ks, "vs": vs}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode_step":
        # the cache as the framework's own prefill of the prompt leaves it
        ctx = case["ctx"]
        shape, model, d = _decoder(case, seed, ctx + 1)
        toks = _tokens(case, seed, ctx + 1)
        nxt = torch.zeros(1, dtype=torch.int32, device=DEV)
        d.prefill(toks[:ctx], 0, nxt, n=ctx)
        return {"kind": kind, "d": d, "model": model, "token": toks[ctx:].clone(), "pos": ctx, "next": nxt}
    if kind == "prompt":
        shape, model, d = _decoder(case, seed, case["N"])
        return {"kind": kind, "d": d, "model": model, "tokens": _tokens(case, seed, case["N"]),
                "next": torch.zeros(1, dtype=torch.int32, device=DEV)}
    s = _inputs(case, seed)
    if kind == "gemv":
        s["y"] = torch.empty(case["M"], dtype=torch.float16, device=DEV)
        s["call"] = _fn("jllm_hip_gemv_quant", s["y"], s["W"], case["type"], s["x"], case["M"], case["K"])
    elif kind == "head":
        s["y"] = torch.empty(case["M"], dtype=torch.float32, device=DEV)
        s["call"] = _fn("jllm_hip_gemv_quant_f32_rmsnorm", s["y"], s["W"], case["type"], s["x"], s["norm"], 1, EPS,
                        case["M"], case["K"])
    elif kind == "gemm":
        s["y"] = torch.empty((case["N"], case["M"]), dtype=torch.float16, device=DEV)
        s["call"] = _fn("jllm_hip_gemm_quant_batched", s["y"], s["W"], case["type"], s["x"], case["M"], case["N"],
                        case["K"])
    else:
        H, kv, hd, i8 = case["heads"], case["kv"], case["hd"], 1 if case["int8"] else 0
        s["y"] = torch.empty_like(s["q"])
        scale = 1.0 / float(np.sqrt(hd))
        if kind == "attn_decode":
            s["call"] = _fn("jllm_hip_flash_attention_decode", s["y"], s["q"], s["k"], s["v"], H, kv, hd, hd,
                            case["ctx"], scale, i8, s["ks"], s["vs"], case["window"])
        else:
            s["call"] = _fn("jllm_hip_flash_attention_prefill_batched", s["y"], s["q"], s["k"], s["v"], H, kv, hd, hd,
                            case["N"], case["start"], scale, i8, s["ks"], s["vs"], case["window"])
    s["kind"] = kind
    return s


def run(state):
    kind = state["kind"]
    if kind == "decode_step":
        state["d"].step(state["token"], state["pos"], state["next"])
        return state["d"].logits()
    if kind == "prompt":
        state["d"].prefill(state["tokens"], 0, state["next"])
        return state["d"].logits()
    f, args, name = state["call"]
    jllm.check(f(*args), name)
    return state["y"]


# ---- work -------------------------------------------------------------------------

def _layer_mats(layer):
    t = decoder.q4km_types(None, layer)
    s = decoder.Shape()
    return [(t[m],) + s.mat_shape(m) for m in decoder.MATS]


def _keys(n, start, window):
    """Sum over n query tokens at positions start.. of the keys each one sees."""
    if window <= 0:
        return n * start + n * (n + 1) // 2
    return sum(min(start + t + 1, window) for t in range(n))


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "head", "gemm"):
        N, M, K, t = case.get("N", 1), case["M"], case["K"], case["type"]
        out = 4 if kind == "head" else 2
        return {"bytes": M * K // 256 * BLOCK[t] + 2 * N * K + out * N * M + (4 * K if kind == "head" else 0),
                "flops": 2 * N * M * K}
    if kind in ("attn_decode", "attn_prefill"):
        n = case.get("N", 1)
        start = case["ctx"] - 1 if kind == "attn_decode" else case["start"]
        seen = start + n - max(0, start + 1 - case["window"] if case["window"] > 0 else 0)
        row = case["kv"] * (case["hd"] + 4 if case["int8"] else 2 * case["hd"])
        return {"bytes": 2 * seen * row + 4 * n * case["heads"] * case["hd"],
                "flops": 4 * case["heads"] * case["hd"] * _keys(n, start, case["window"])}
    n, start = (1, case["ctx"]) if kind == "decode_step" else (case["N"], 0)
    by, fl = case["vocab"] * HID // 256 * BLOCK[Q6] + 4 * case["vocab"] + n * HID // 256 * BLOCK[Q4], 2 * case["vocab"] * HID
    for l in range(case["layers"]):
        for t, M, K in _layer_mats(l):
            by += M * K // 256 * BLOCK[t]
            fl += 2 * n * M * K
        by += 2 * (start + n) * KV * (HD + 4)
        fl += 4 * HEADS * HD * _keys(n, start, 0)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """Largest relative error of another correct implementation at the same precision:
    about four times what the same inputs show with the sums in another order."""
    kind = case["kind"]
    if kind == "head":
        return {"rel": 4e-4, "max": 2e-2}     # fp32 sums; single fp16 roundings of the normalised activation differ
    if kind == "gemm":
        # fp16 outputs; the products of a block's fp16 scales and 6-bit sub-scales are
        # rounded to fp16, or kept, as an implementation likes: 2e-4
        return {"rel": 1e-3, "max": 2e-2}
    if kind in ("gemv", "attn_decode", "attn_prefill"):
        return {"rel": 1e-3, "max": 2e-2}     # fp16 outputs: single roundings differ
    # whole calls: the int8 activation and KV codes that sit at a rounding edge move by one
    # code, and every later product sees it
    return {"rel": 3e-2, "max": 3e-1}


# ---- 64-bit results -----------------------------------------------------------------

def _scale_min(s):
    """6-bit scales and mins [..., 8] of the 12 packed bytes of a Q4_K / Q5_K header."""
    s = s.to(torch.int32)
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    return sc.double(), mn.double()


def _parts(W, t, M, K):
    """The two linear parts of the weights in float64: (A [M, K], B [M, K / 32]) with
    w = A - B (B per 32 weights; None for Q6_K)."""
    nb = K // 256
    b = W.view(M, nb, BLOCK[t])

    def f16(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()
    if t == Q6:
        ql, qh = b[..., 0:128].reshape(M, nb, 2, 64), b[..., 128:192].reshape(M, nb, 2, 32)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        q = torch.stack([(ql[..., 0:32] & 15) | ((qh & 3) << 4), (ql[..., 32:64] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., 0:32] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 32:64] >> 4) | ((qh >> 6) << 4)], 3)
        q = q.reshape(M, nb, 16, 16).double() - 32.0
        return (q * (f16(208) * sc)[..., None]).reshape(M, K), None
    sc, mn = _scale_min(b[..., 4:16])
    qs = b[..., BLOCK[t] - 128:].reshape(M, nb, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 3).reshape(M, nb, 8, 32)
    if t == Q5:
        bit = torch.arange(8, device=DEV, dtype=torch.uint8).view(8, 1)
        q = q | (((b[..., None, 16:48] >> bit) & 1) << 4)
    return (q.double() * (f16(0) * sc)[..., None]).reshape(M, K), (f16(2) * mn).reshape(M, K // 32)


def _q8(x, clamp):
    """The path's int8 activation quantisation per 32 values, in its own fp32 arithmetic:
    (codes, d fp32, block sums of x fp32)."""
    v = x.float().view(x.shape[0], -1, 32)
    d = v.abs().amax(-1) / torch.full((), 127.0, device=DEV)
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    q = torch.round(v * inv[..., None])
    if clamp:
        q = q.clamp(-127, 127)
    return q, d, v.sum(-1)


def _product(W, t, M, K, x, mode):
    """W . x in float64 with the activation as the path takes it: mode "mmq" (prefill),
    "mmvq" (decode) quantise it to int8 blocks first, "float" takes the fp16 values."""
    y = torch.empty((x.shape[0], M), dtype=torch.float64, device=DEV)
    if mode == "float":
        a, s = x.double(), x.double().view(x.shape[0], -1, 32).sum(-1)
    else:
        q, d, sx = _q8(x, mode == "mmvq")
        dh = d if (t == Q6 and mode == "mmq") else d.half().float()
        a = (q.double() * dh.double()[..., None]).reshape(x.shape)
        s = (sx if mode == "mmq" else d * q.sum(-1)).half().double()
    step = max(1, (1 << 27) // K)
    for r in range(0, M, step):
        A, B = _parts(W.view(M, -1)[r:r + step], t, min(step, M - r), K)
        y[:, r:r + step] = a @ A.t()
        if B is not None:
            y[:, r:r + step] -= s @ B.t()
    return y


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, k, v, start, window):
    """Causal attention in float64: q [n, H, hd] at positions start.., k / v [ctx, kv, hd]."""
    n, H, hd = q.shape
    ctx, kv = k.shape[0], k.shape[1]
    pos, key = torch.arange(start, start + n, device=DEV)[:, None], torch.arange(ctx, device=DEV)[None, :]
    dead = key > pos
    if window > 0:
        dead = dead | (key <= pos - window)
    out = torch.empty_like(q)
    for h in range(H):
        g = h // (H // kv)
        for r in range(0, n, 1024):
            s = (q[r:r + 1024, h] @ k[:, g].t().contiguous()) / hd ** 0.5
            out[r:r + 1024, h] = torch.softmax(s.masked_fill(dead[r:r + 1024], float("-inf")), -1) @ v[:, g].contiguous()
    return out


def _model_logits(case, model, tokens):
    """The decoder in float64 over the dequantised weights, nothing quantised or rounded
    in between: the logits of the last token."""
    def mat(L, m):
        M, K = decoder.Shape().mat_shape(m)
        return lambda x: _product(L[m], L["types"][m], M, K, x, "float")
    n = tokens.numel()
    rows = model["tok_embd"].view(case["vocab"], -1)[tokens.long()].contiguous()
    A, B = _parts(rows, Q4, n, HID)
    x = A - B.repeat_interleave(32, -1)
    inv = decoder.Shape().rope_theta ** (-torch.arange(0, HD, 2, device=DEV).double() / HD)
    ang = torch.arange(n, device=DEV).double()[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(v):
        a, b = v[..., :HD // 2], v[..., HD // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)
    for L in model["layers"]:
        h = _rms(x, L["rms_attn"])
        q = rope(_rms(mat(L, "wq")(h).view(n, HEADS, HD), L["q_norm"]))
        k = rope(_rms(mat(L, "wk")(h).view(n, KV, HD), L["k_norm"]))
        v = mat(L, "wv")(h).view(n, KV, HD)
        x = x + mat(L, "wo")(_attend(q, k, v, 0, 0).reshape(n, QD))
        h = _rms(x, L["rms_ffn"])
        g = mat(L, "w_gate")(h)
        x = x + mat(L, "w_down")(g * torch.sigmoid(g) * mat(L, "w_up")(h))
    h = _rms(x[-1:], model["output_norm"])
    return _product(model["output"], Q6, case["vocab"], HID, h, "float").view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode_step", "prompt"):
        n = case["ctx"] + 1 if kind == "decode_step" else case["N"]
        shape = decoder.Shape(n_layers=case["layers"], vocab_size=case["vocab"])
        return _model_logits(case, decoder.synth_device(shape, int(seed), DEV), _tokens(case, seed, n))
    s = _inputs(case, seed)
    if kind in ("gemv", "head", "gemm"):
        t, M, K = case["type"], case["M"], case["K"]
        if kind == "gemm":
            return _product(s["W"], t, M, K, s["x"], "float" if t == Q5 else "mmq")
        if kind == "gemv":
            return _product(s["W"], t, M, K, s["x"], "float" if t == Q5 else "mmvq").view(-1)
        x = _rms(s["x"].double(), s["norm"]).half()
        return _product(s["W"], t, M, K, x, "float" if t == Q6 else "mmvq").view(-1)
    k, v = s["k"].double(), s["v"].double()
    if case["int8"]:
        k, v = k * s["ks"].double()[..., None], v * s["vs"].double()[..., None]
    start = case["ctx"] - 1 if kind == "attn_decode" else case["start"]
    return _attend(s["q"].double(), k, v, start, case["window"])
