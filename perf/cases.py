"""The work this framework is used for, as cases that can be timed and compared.

Each case is one call (or one turn of a generation session) through the public entry points of
include/af.h, as adaforge_amd's bindings expose them: the Q4_0 GEMV and batched GEMV, the FFN block,
the Q6_K head with greedy selection, decode attention over the fp16 cache, and whole sessions
(prompt prefill, greedy decode, the logits after a further token).  Shapes are those of the
12B-shaped model the benchmark decodes and of the test models; the ranges `draw` spreads over reach
from a few rows to the largest matrices of that model.

Inputs come from the seed alone and are made on the GPU: Q4_0 matrices are Gaussian weights put
through GGUF's quantiser (d = the largest weight / -8), Q6_K tables have uniform codes, activations
and cached K/V are N(0, 1).
"""
import ctypes
import math

import numpy as np
import torch

from adaforge_amd import _native as N
from adaforge_amd.backend import HipDiagnostics
from adaforge_amd.synth import SynthLayer, SynthModel, gemma4_rope_factors

DEV = "cuda"
EPS = 1e-6
VOCAB = 32768      # of the session cases
ROPE_CONTEXT = 131072


# ---- the cases ---------------------------------------------------------------------------------

def _gemv(rows, columns):
    return {"kind": "gemv", "rows": rows, "columns": columns}


def _gemm(tokens, rows, columns):
    return {"kind": "gemm", "tokens": tokens, "rows": rows, "columns": columns}


def _ffn(hidden, intermediate, post):
    return {"kind": "ffn", "hidden": hidden, "intermediate": intermediate, "post": post}


def _head(rows, columns):
    return {"kind": "head", "rows": rows, "columns": columns}


def _attention(context, window, q_heads, kv_heads, width):
    return {"kind": "attention", "context": context, "window": window, "q_heads": q_heads, "kv_heads": kv_heads,
            "width": width}


def _session(shape, layers, prompt, new, window):
    return {"kind": "session", "shape": shape, "layers": layers, "prompt": prompt, "new": new, "window": window}


def listed():
    return [
        # one attention-query projection for one token: the smallest call of the path
        dict(_gemv(4096, 3840), name="gemv_4096x3840"),
        # a matrix whose rows and columns are multiples of nothing the kernels tile by
        dict(_gemv(1001, 2080), name="gemv_1001x2080"),
        # a full batch of prompt tokens through an FFN gate
        dict(_gemm(32, 15360, 3840), name="gemm_32_15360x3840"),
        # a short speculative draft through the FFN's down projection
        dict(_gemm(5, 3840, 15360), name="gemm_5_3840x15360"),
        # the feed-forward block of one token
        dict(_ffn(3840, 15360, False), name="ffn_3840x15360"),
        # vocabulary logits and the greedy id: the largest single read of a token
        dict(_head(262144, 3840), name="head_262144x3840"),
        # one token's attention early in a conversation, in a sliding-window layer
        dict(_attention(512, 1024, 16, 8, 256), name="attention_local_512"),
        # one token's attention in a global layer at the longest context
        dict(_attention(32768, 0, 16, 8, 256), name="attention_global_32768"),
        # a global layer of the Gemma-4-shaped model: 16 query heads share one 512-wide KV head
        dict(_attention(4096, 0, 16, 1, 512), name="attention_512wide_4096"),
        # the first turn on a long prompt: prefill bound
        dict(_session("gemma3", 6, 512, 1, 1024), name="session_prefill_512"),
        # a short question with a longer answer: decode bound
        dict(_session("gemma3", 6, 24, 64, 1024), name="session_decode_64"),
        # a long document into the Gemma-4-shaped model (past its window), then a short answer
        dict(_session("gemma4", 6, 1500, 32, 1024), name="session_gemma4_1500"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "gemm", "ffn", "head", "attention", "attention", "session", "session"])
    if kind == "gemv":
        return _gemv(_log(rng, 200, 15360), 32 * _log(rng, 16, 480))
    if kind == "gemm":
        return _gemm(rng.randint(1, 32), _log(rng, 200, 15360), 32 * _log(rng, 16, 480))
    if kind == "ffn":
        return _ffn(32 * rng.randint(16, 120), 32 * _log(rng, 32, 480), rng.random() < 0.5)
    if kind == "head":
        return _head(_log(rng, 1000, 262144), 256 * rng.randint(2, 15))
    if kind == "attention":
        context = _log(rng, 16, 32768)
        window = rng.choice([0, 0, 512, 1024])
        if rng.random() < 0.7:
            kv = rng.choice([1, 2, 4, 8])
            return _attention(context, window, kv * rng.choice([1, 2, 4]), kv, 256)
        return _attention(min(context, 16384), window, rng.choice([4, 8, 16]), 1, 512)
    return _session(rng.choice(["gemma3", "gemma3", "gemma4"]), rng.randint(2, 6), _log(rng, 2, 1500), _log(rng, 1, 32),
                    rng.choice([512, 1024]))


# ---- seeded inputs -----------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _q4(g, rows, columns, sigma=0.02):
    """GGUF Q4_0 bytes [rows * columns / 32][18] of N(0, sigma) weights."""
    w = _randn(g, rows * (columns // 32), 32) * sigma
    m = w.gather(1, w.abs().argmax(1, keepdim=True))
    d = (m / -8).half()
    n = torch.clamp(torch.floor(w / d.float() + 8.5), 0, 15).to(torch.uint8)
    return torch.cat([d.view(torch.uint8), n[:, :16] | (n[:, 16:] << 4)], 1)


def _q6(g, rows, columns, low, high):
    """GGUF Q6_K bytes [rows * columns / 256][210]: uniform codes, sub-scales in [-32, 31], d in [low, high]."""
    n = rows * (columns // 256)
    out = torch.randint(0, 256, (n, 210), generator=g, device=DEV, dtype=torch.uint8)
    out[:, 192:208] = torch.randint(-32, 32, (n, 16), generator=g, device=DEV, dtype=torch.int8).view(torch.uint8)
    d = torch.rand(n, 1, generator=g, device=DEV) * (high - low) + low
    out[:, 208:] = d.half().view(torch.uint8)
    return out


def _host(b):
    return b.cpu().numpy().reshape(-1)


def _norm(g, n):
    return 1.0 + 0.1 * _randn(g, n)


def _bytes_args(a):
    return a.ctypes.data_as(N.u8p), a.size


def _operator(case, seed):
    """The inputs of an operator case, as GPU tensors."""
    g, k = _generator(seed), case["kind"]
    if k in ("gemv", "gemm"):
        return {"w": _q4(g, case["rows"], case["columns"]), "x": _randn(g, case.get("tokens", 1), case["columns"])}
    if k == "ffn":
        h, i = case["hidden"], case["intermediate"]
        return {"gate": _q4(g, i, h), "up": _q4(g, i, h), "down": _q4(g, h, i), "pre": _norm(g, h),
                "post": _norm(g, h) if case["post"] else None, "scale": 0.75 if case["post"] else 1.0,
                "x": _randn(g, h)}
    if k == "head":
        return {"w": _q6(g, case["rows"], case["columns"], 1e-4, 5e-3), "x": _randn(g, case["columns"])}
    ring = _ring(case)
    kv, w = case["kv_heads"], case["width"]
    return {"q": _randn(g, case["q_heads"], w), "k": _randn(g, kv, w), "v": _randn(g, kv, w), "q_norm": _norm(g, w),
            "k_norm": _norm(g, w), "k_cache": _randn(g, kv, ring, w).half(), "v_cache": _randn(g, kv, ring, w).half()}


def _ring(case):
    return min(case["window"] + 32, case["context"]) if case["window"] else case["context"]


def _rope(case):
    """Base and frequency divisors: a global 512-wide layer turns only its first 64 pairs."""
    if case["width"] == 512:
        return 1e6, gemma4_rope_factors(512)
    return (1e4 if case["window"] else 1e6), np.ones(case["width"] // 2, np.float32)


def _model(case, seed):
    """Weights of a session case: GPU tensors in SynthLayer's fields, the Q6_K table, the prompt.

    The table's scale gives the input token's own logit a lead over the others, as wide as a trained
    model's usual one, so that the greedy ids do not hang on the last bits of a logit while the
    residual stream still comes mostly from the layers."""
    g = _generator(seed)
    H, I = 3840, 15360
    layers = []
    for i in range(case["layers"]):
        glob = i % 6 == 5 or (case["layers"] < 6 and i == case["layers"] - 1)
        g4 = case["shape"] == "gemma4"
        qh, kvh, hw = (16, 1, 512) if g4 and glob else (16, 8, 256)
        # a score scale of 1 goes with query norms that hold the 1 / sqrt(width)
        q_norm = _norm(g, hw) * (hw ** -0.5 if g4 else 1.0)
        layers.append(SynthLayer(
            input_norm=_norm(g, H), q=_q4(g, qh * hw, H), k=_q4(g, kvh * hw, H),
            v=None if g4 and glob else _q4(g, kvh * hw, H), q_norm=q_norm, k_norm=_norm(g, hw),
            rope_base=1e6 if glob else 1e4,
            rope_factors=gemma4_rope_factors(hw) if g4 and glob else np.ones(hw // 2, np.float32),
            rope_context=ROPE_CONTEXT, q_heads=qh, kv_heads=kvh, head_width=hw, window=None if glob else case["window"],
            scale=1.0 if g4 else 1.0 / 16.0, o=_q4(g, H, qh * hw), post_attn_norm=_norm(g, H), ffn_norm=_norm(g, H),
            gate=_q4(g, I, H), up=_q4(g, I, H), down=_q4(g, H, I), post_ffn_norm=_norm(g, H), eps=EPS, v_norm=g4))
    ids = torch.randint(0, VOCAB - 1, (case["prompt"] + 1,), generator=g, device=DEV).cpu().numpy().astype(np.uint32)
    return SynthModel(hidden=H, intermediate=I, vocabulary=VOCAB, table=_q6(g, VOCAB, H, 1e-5, 8e-5),
                      final_norm=_norm(g, H), final_eps=EPS, layers=layers), ids


def prepare(case, seed):
    k = case["kind"]
    if k == "session":
        model, ids = _model(case, seed)
        for L in model.layers:
            for f in ("q", "k", "v", "o", "gate", "up", "down"):
                if getattr(L, f) is not None:
                    setattr(L, f, _host(getattr(L, f)))
            for f in ("input_norm", "q_norm", "k_norm", "post_attn_norm", "ffn_norm", "post_ffn_norm"):
                setattr(L, f, getattr(L, f).cpu().numpy())
        model.table, model.final_norm = _host(model.table), model.final_norm.cpu().numpy()
        torch.cuda.empty_cache()
        session = HipDiagnostics().open_session(model, case["prompt"] + case["new"] + 8)
        session._keep.items.clear()  # the session owns device copies; the host weights may go
        return {"kind": k, "session": session, "prompt": ids[:-1], "follow": ids[-1:], "new": case["new"]}
    t = _operator(case, seed)
    s = {"kind": k, "stream": torch.cuda.current_stream().cuda_stream, "lib": N.lib()}
    if k in ("gemv", "gemm"):
        w, h = _host(t["w"]), N.P()
        N.check(N.lib().af_q4_upload(*_bytes_args(w), case["columns"], case["rows"], ctypes.byref(h)))
        s.update(w=_Handle(h, N.lib().af_q4_free), x=t["x"], tokens=case.get("tokens", 1),
                 y=torch.empty(case.get("tokens", 1), case["rows"], device=DEV))
    elif k == "ffn":
        H, I = case["hidden"], case["intermediate"]
        keep = {f: _host(t[f]) for f in ("gate", "up", "down")}
        keep.update({f: t[f].cpu().numpy() for f in ("pre", "post") if t[f] is not None})

        def norm(f):
            return N.RmsNormDesc(keep[f].ctypes.data_as(N.f32p), H, EPS) if f in keep else N.RmsNormDesc(None, 0, EPS)

        d = N.FfnDesc(norm("pre"), N.MatrixDesc(*_bytes_args(keep["gate"]), H, I),
                      N.MatrixDesc(*_bytes_args(keep["up"]), H, I), N.MatrixDesc(*_bytes_args(keep["down"]), I, H),
                      norm("post"), t["scale"])
        h = N.P()
        N.check(N.lib().af_ffn_create(ctypes.byref(d), ctypes.byref(h)))
        s.update(w=_Handle(h, N.lib().af_ffn_free), x=t["x"], y=torch.empty(H, device=DEV))
    elif k == "head":
        w, h = _host(t["w"]), N.P()
        N.check(N.lib().af_q6_upload(*_bytes_args(w), case["columns"], case["rows"], ctypes.byref(h)))
        s.update(w=_Handle(h, N.lib().af_q6_free), x=t["x"], y=torch.empty(case["rows"], device=DEV),
                 result=torch.empty(2, dtype=torch.int32, device=DEV))
    else:
        base, factors = _rope(case)
        s.update(t, factors=factors, y=torch.empty(case["q_heads"], case["width"], device=DEV))
        p = lambda n: t[n].data_ptr()  # noqa: E731
        s["args"] = N.AttentionArgs(
            p("q"), p("k"), p("v"), p("q_norm"), p("k_norm"), EPS, EPS, EPS, 1 if case["width"] == 512 else 0,
            N.RopeDesc(case["width"], base, factors.ctypes.data_as(N.f32p), ROPE_CONTEXT),
            N.AttentionConfigDesc(case["q_heads"], case["kv_heads"], case["width"], case["window"], _scale(case)),
            p("k_cache"), p("v_cache"), _ring(case), case["context"] - 1, s["y"].data_ptr())
    return s


def _scale(case):
    return 1.0 / math.sqrt(case["width"])


class _Handle:
    """A device-resident matrix or block, freed with the state that holds it."""

    def __init__(self, h, free):
        self.h, self.free = h, free

    def __del__(self):
        self.free(self.h)


def run(s):
    k = s["kind"]
    if k == "session":
        # a turn from an empty cache: the prompt, the greedy ids, then the logits after one more token
        session = s["session"]
        session.reset()
        got = session.generate(s["prompt"], [VOCAB - 1], s["new"])
        _, _, logits, hidden = session.trace(s["follow"], layer_outputs=False)
        return {"ids": np.asarray(got.ids, np.int64), "logits": logits, "hidden": hidden}
    lib, stream = s["lib"], s["stream"]
    if k == "gemv":
        N.check(lib.af_q4_gemv(s["w"].h, s["x"].data_ptr(), s["y"].data_ptr(), stream))
        return s["y"]
    if k == "gemm":
        N.check(lib.af_q4_gemm(s["w"].h, s["x"].data_ptr(), s["tokens"], s["y"].data_ptr(), stream))
        return s["y"]
    if k == "ffn":
        N.check(lib.af_ffn_run(s["w"].h, s["x"].data_ptr(), s["y"].data_ptr(), stream))
        return s["y"]
    if k == "head":
        N.check(lib.af_q6_gemv_argmax(s["w"].h, s["x"].data_ptr(), s["y"].data_ptr(), s["result"].data_ptr(), stream))
        return {"logits": s["y"], "result": s["result"]}
    N.check(lib.af_attention_decode(ctypes.byref(s["args"]), stream))
    return {"out": s["y"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


# ---- what a pass cannot do without ---------------------------------------------------------------

def _q4_bytes(rows, columns):
    return rows * (columns // 32) * 18


def work(case):
    k = case["kind"]
    if k in ("gemv", "gemm"):
        r, c, t = case["rows"], case["columns"], case.get("tokens", 1)
        return {"bytes": _q4_bytes(r, c) + 4 * t * (r + c), "flops": 2 * r * c * t}
    if k == "ffn":
        h, i = case["hidden"], case["intermediate"]
        return {"bytes": 3 * _q4_bytes(h, i) + 8 * h, "flops": 6 * h * i}
    if k == "head":
        r, c = case["rows"], case["columns"]
        return {"bytes": r * (c // 256) * 210 + 4 * (r + c), "flops": 2 * r * c}
    if k == "attention":
        n = min(case["context"], case["window"] or case["context"])
        return {"bytes": n * case["kv_heads"] * case["width"] * 4 + 8 * case["q_heads"] * case["width"],
                "flops": 4 * n * case["q_heads"] * case["width"]}
    H, I, P = 3840, 15360, case["prompt"]
    steps = case["new"] + 1          # tokens decoded one at a time: the prompt's last, the ids, the further one
    total = P + steps
    weights = weight_bytes = cache_bytes = flops = 0
    for i in range(case["layers"]):
        glob = i % 6 == 5 or (case["layers"] < 6 and i == case["layers"] - 1)
        qd, kd = (8192, 512) if glob and case["shape"] == "gemma4" else (4096, 2048)
        sets = 1 if glob and case["shape"] == "gemma4" else 2
        n = H * (2 * qd + sets * kd + 3 * I)
        weights += n
        weight_bytes += n // 32 * 18
        span = lambda p: p + 1 if glob else min(p + 1, case["window"])  # noqa: E731
        flops += 4 * qd * sum(span(p) for p in range(total))
        cache_bytes += 4 * kd * (total + sum(span(p) for p in range(P - 1, total)))
    head = VOCAB * H
    prefill = 1 if P > 1 else 0
    return {"bytes": (prefill + steps + 1) * weight_bytes + (steps + 1) * head // 256 * 210 + cache_bytes,
            "flops": flops + 2 * weights * total + 2 * head * (steps + 1)}


# ---- tolerances and the 64-bit answers -------------------------------------------------------------

def tolerance(case):
    k = case["kind"]
    # four times what is seen against the 64-bit answers: 32-bit sums over up to 15360 columns
    if k in ("gemv", "gemm", "head"):
        return {"rel": 1e-6, "max": 2e-5, "differ": 0.0}
    if k == "ffn":
        return {"rel": 2e-6, "max": 4e-5}
    if k == "attention":
        # 32-bit softmax and sums; the appended K and V are fp16, where one ulp may differ
        return {"rel": 2e-6, "max": 1.1e-3}
    # several layers, whose fp16 K and V round to the neighbouring value where 32-bit sums differ
    return {"rel": 3e-4, "max": 2e-3, "differ": 0.0}


def _deq4(b, rows, columns):
    d = b[:, :2].contiguous().view(torch.float16).double()
    n = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0
    return (n * d).reshape(rows, columns)


def _deq6(b, rows, columns):
    """rows x columns doubles of GGUF Q6_K super-blocks."""
    n = b.shape[0]
    d = b[:, 208:].contiguous().view(torch.float16).double()
    sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
    ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
    code = torch.stack([(ql[:, :, q % 2] >> (4 * (q // 2)) & 15) | ((qh >> (2 * q) & 3) << 4) for q in range(4)], 2)
    w = (code.double() - 32.0).reshape(n, 2, 4, 2, 16) * sc * d.reshape(n, 1, 1, 1, 1)
    return w.reshape(rows, columns)


def _rms(x, w, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x * x * x)))


def _rotate(x, base, factors, pos):
    """NeoX RoPE of x [tokens][heads][width] at positions pos [tokens]."""
    half = x.shape[-1] // 2
    i = torch.arange(half, device=DEV, dtype=torch.float64)
    f = base ** (-2.0 * i / (2 * half)) / torch.as_tensor(factors, device=DEV).double()
    a = pos.double()[:, None, None] * f
    s, c = torch.sin(a), torch.cos(a)
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, u * s + v * c], -1)


def _attend(q, k, v, scale, pos, window):
    """q [T][qh][w] at positions pos over k, v [n][kvh][w] (rows are positions 0 .. n - 1)."""
    T, qh, w = q.shape
    n, kvh, _ = k.shape
    out = torch.empty_like(q)
    keys = torch.arange(n, device=DEV)
    seen = keys[None] <= pos[:, None]
    if window:
        seen &= keys[None] > pos[:, None] - window
    for h in range(qh):
        s = (q[:, h] @ k[:, h * kvh // qh].t()) * scale
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ v[:, h * kvh // qh]
    return out


def _exact_attention(case, t):
    base, factors = _rope(case)
    pos = torch.tensor([case["context"] - 1], device=DEV)
    f64 = {n: x.double() for n, x in t.items()}
    q = _rotate(_rms(f64["q"], f64["q_norm"])[None], base, factors, pos)
    k = _rotate(_rms(f64["k"], f64["k_norm"])[None], base, factors, pos)[0]
    v = _rms(f64["v"], 1.0) if case["width"] == 512 else f64["v"]
    slot = (case["context"] - 1) % _ring(case)
    kc, vc = f64["k_cache"], f64["v_cache"]
    kc[:, slot], vc[:, slot] = k.float().half().double(), v.float().half().double()
    first = max(0, case["context"] - case["window"]) if case["window"] else 0
    at = torch.arange(first, case["context"], device=DEV) % _ring(case)
    out = _attend(q, kc[:, at].transpose(0, 1), vc[:, at].transpose(0, 1), _scale(case),
                  torch.tensor([at.numel() - 1], device=DEV), 0)
    return {"out": out[0], "k_cache": kc, "v_cache": vc}


def _exact_session(case, seed):
    """The turn in 64 bits throughout, the cached K and V too (the framework's cache is fp16)."""
    model, ids = _model(case, seed)
    H = model.hidden
    table = _deq6(model.table, VOCAB, H)
    dense, caches = [], []
    for L in model.layers:
        qd, kd = L.q_heads * L.head_width, L.kv_heads * L.head_width
        shapes = {"q": (qd, H), "k": (kd, H), "v": (kd, H), "o": (H, qd), "gate": (15360, H), "up": (15360, H),
                  "down": (H, 15360)}
        W = {f: _deq4(getattr(L, f), *s) for f, s in shapes.items() if getattr(L, f) is not None}
        W.update({f: getattr(L, f).double() for f in ("input_norm", "q_norm", "k_norm", "post_attn_norm", "ffn_norm",
                                                      "post_ffn_norm")})
        dense.append(W)
        caches.append([torch.empty(0, L.kv_heads, L.head_width, device=DEV, dtype=torch.float64) for _ in range(2)])

    def forward(tokens, p0):
        pos = torch.arange(p0, p0 + len(tokens), device=DEV)
        x = table[torch.as_tensor(np.asarray(tokens, np.int64), device=DEV)] * math.sqrt(H)
        for L, W, C in zip(model.layers, dense, caches):
            n, T = _rms(x, W["input_norm"]), len(tokens)
            heads = lambda y: y.reshape(T, -1, L.head_width)  # noqa: E731
            kr = heads(n @ W["k"].t())
            q = _rotate(_rms(heads(n @ W["q"].t()), W["q_norm"]), L.rope_base, L.rope_factors, pos)
            k = _rotate(_rms(kr, W["k_norm"]), L.rope_base, L.rope_factors, pos)
            v = heads(n @ W["v"].t()) if L.v is not None else kr
            if L.v_norm:
                v = _rms(v, 1.0)
            C[0], C[1] = torch.cat([C[0], k]), torch.cat([C[1], v])
            a = _attend(q, C[0], C[1], L.scale, pos, L.window or 0).reshape(T, -1)
            x = x + _rms(a @ W["o"].t(), W["post_attn_norm"])
            n = _rms(x, W["ffn_norm"])
            x = x + _rms((_gelu(n @ W["gate"].t()) * (n @ W["up"].t())) @ W["down"].t(), W["post_ffn_norm"])
        return x[-1]

    def logits_of(h):
        return table @ _rms(h, model.final_norm.double())

    h, p, got = forward(ids[:-1], 0), case["prompt"], []
    for _ in range(case["new"]):
        got.append(int(torch.argmax(logits_of(h))))
        if got[-1] == VOCAB - 1:
            got.pop()
            break
        h = forward(got[-1:], p)
        p += 1
    h = forward(ids[-1:], p)
    return {"ids": None, "logits": logits_of(h), "hidden": h}


def exact(case, seed):
    k = case["kind"]
    if k == "session":
        return _exact_session(case, seed)
    t = _operator(case, seed)
    if k in ("gemv", "gemm"):
        return t["x"].double() @ _deq4(t["w"], case["rows"], case["columns"]).t()
    if k == "ffn":
        h, i = case["hidden"], case["intermediate"]
        x = t["x"].double()
        n = _rms(x, t["pre"].double())
        a = _gelu(_deq4(t["gate"], i, h) @ n) * (_deq4(t["up"], i, h) @ n)
        d = _deq4(t["down"], h, i) @ a
        if t["post"] is not None:
            d = _rms(d, t["post"].double())
        return (d + x) * t["scale"]
    if k == "head":
        r, c = case["rows"], case["columns"]
        per, x = c // 256, t["x"].double()
        parts = [_deq6(t["w"][a * per:min(a + 16384, r) * per], min(a + 16384, r) - a, c) @ x for a in range(0, r, 16384)]
        return {"logits": torch.cat(parts), "result": None}
    return _exact_attention(case, t)
