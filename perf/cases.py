"""Performance cases: what a program that uses this library has it do.

Each case is one call (or one whole engine call) through the public entry
points, at the shapes of the two models the library serves: the E4B-shaped
decoder (hidden 2048, FFN 16384, 8 q / 2 KV heads of 256, per-layer
embeddings, Q6_K head of 262144 rows) and the A4B mixture of experts (hidden
2816, 128 experts of 704, dense branch 2112).  Sizes in between are drawn:
ragged prompt lengths, odd row counts, other cache positions.

Kinds:
  gemv         q4_0 matrix x one vector (decode)              e4b_k_q40_gemv
  lmhead       Q6_K head + softcap + argmax (decode)          e4b_k_q6k_gemv_argmax
  attn_decode  one layer's attention of one token (decode)    e4b_k_attn_decode
  moe          one MoE half-layer of one token (decode)       e4b_k_moe_layer
  gemm         q4_0 matrix x m token rows (prefill)           e4b_k_q40_gemm
  geglu        gate/up + GeGLU over m token rows (prefill)    e4b_k_q40_gemm_geglu
  attn_prefill causal attention of a prompt chunk (prefill)   e4b_k_attn_prefill
  moe_prefill  one MoE half-layer over m tokens (prefill)     e4b_k_moe_prefill
  prompt       an E4B-shaped engine's batched prefill         Engine.prefill
  steps        the same engine, token by token (decode step)  Engine.prefill_steps
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "e4b-webgpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

EPS = 1e-6
SOFTCAP = 30.0
HEAD_DIM = 256
LAYERS = 5         # of the engine cases: four sliding layers and a global one, as one period of the model
MAX_SEQ = 2048
TOP_K = 8

# q4_0 matrices of the two models (rows, cols)
MATRICES = [(256, 2048), (2048, 256), (3072, 2048), (2048, 2048), (2048, 16384), (8960, 2048), (16384, 2048),
            (32768, 2048), (8192, 2816), (9216, 2816), (2816, 4096), (2816, 8192), (4224, 2816), (2816, 2112)]


def listed():
    return [
        # the per-layer-embedding gate of one decoded token: the smallest matrix of a step, all latency
        {"name": "gemv_256x2048_f16", "kind": "gemv", "rows": 256, "cols": 2048, "f16": True},
        # one half of the FFN input projection for one token, f32 activations: an ordinary decode GEMV
        {"name": "gemv_16384x2048_f32", "kind": "gemv", "rows": 16384, "cols": 2048, "f16": False},
        # the head of every decoded token: the largest single matrix of a step
        {"name": "lmhead_262144x2048", "kind": "lmhead", "rows": 262144, "cols": 2048},
        # a global layer's attention of one token, late in a 4096-token context
        {"name": "attn_decode_global_4095", "kind": "attn_decode", "slots": 4096, "window": 0, "pos": 4095},
        # one MoE half-layer of one decoded token
        {"name": "moe_layer", "kind": "moe", "hidden": 2816, "experts": 128, "ff": 704, "dense": 2112},
        # q|k|v of a short chat turn: a ragged handful of tokens
        {"name": "gemm_3072x2048_m37", "kind": "gemm", "rows": 3072, "cols": 2048, "m": 37},
        # the FFN output projection of a full prompt chunk: the longest reduction
        {"name": "gemm_2048x16384_m512", "kind": "gemm", "rows": 2048, "cols": 16384, "m": 512},
        # the FFN input projection + GeGLU of a full prompt chunk: most of a prompt's work
        {"name": "geglu_16384x2048_m512", "kind": "geglu", "ff": 16384, "cols": 2048, "m": 512},
        # a sliding layer's attention of the second chunk of a prompt (the window is full)
        {"name": "attn_prefill_sliding_512", "kind": "attn_prefill", "m": 512, "p0": 512, "window": 512,
         "slots": 1024, "q_heads": 8, "kv_heads": 2},
        # one MoE half-layer over a full prompt chunk
        {"name": "moe_prefill_512", "kind": "moe_prefill", "hidden": 2816, "experts": 128, "ff": 704,
         "dense": 2112, "m": 512},
        # a 512-token prompt through the engine, to the logits of its last token
        {"name": "prompt_512", "kind": "prompt", "n": 512},
        # 96 tokens through the decode step, to the logits of the last one
        {"name": "steps_96", "kind": "steps", "n": 96},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemv", "lmhead", "attn_decode", "moe", "gemm", "gemm", "geglu", "attn_prefill", "moe_prefill",
                       "prompt", "steps"])
    if kind == "gemv":
        rows, cols = rng.choice(MATRICES)
        if rng.random() < 0.5:  # a matrix of another model
            rows, cols = _log(rng, 37, 32768), 32 * _log(rng, 3, 128)
        return {"kind": kind, "rows": rows, "cols": cols, "f16": rng.random() < 0.5}
    if kind == "lmhead":
        return {"kind": kind, "rows": _log(rng, 1000, 262143), "cols": rng.choice([256, 512, 1024, 2048, 2816])}
    if kind == "attn_decode":
        if rng.random() < 0.5:
            return {"kind": kind, "slots": 1024, "window": 512, "pos": _log(rng, 1, 8191)}
        pos = _log(rng, 1, 8191)
        return {"kind": kind, "slots": pos + 1 + rng.randrange(64), "window": 0, "pos": pos}
    if kind == "moe" or kind == "moe_prefill":
        c = {"kind": kind, "hidden": rng.choice([1024, 2048, 2816]), "experts": rng.choice([16, 61, 64, 128]),
             "ff": 32 * rng.randint(4, 22), "dense": 32 * rng.randint(16, 66)}
        if kind == "moe_prefill":
            c["m"] = _log(rng, 1, 512)
        return c
    if kind == "gemm":
        rows, cols = rng.choice(MATRICES)
        if rng.random() < 0.4:
            rows, cols = _log(rng, 37, 16384), 32 * _log(rng, 3, 128)
        return {"kind": kind, "rows": rows, "cols": cols, "m": _log(rng, 1, 512)}
    if kind == "geglu":
        ff, cols = rng.choice([(16384, 2048), (2112, 2816), (704, 2816)])
        if rng.random() < 0.4:
            ff, cols = _log(rng, 100, 16384), 32 * _log(rng, 8, 64)
        return {"kind": kind, "ff": ff, "cols": cols, "m": _log(rng, 1, 512)}
    if kind == "attn_prefill":
        kvh = rng.choice([1, 2, 8])
        qh = kvh * (2 if kvh == 8 else rng.choice([2, 4]))
        m = _log(rng, 1, 512)
        p0 = rng.choice([0, _log(rng, 1, 3584)])
        if rng.random() < 0.5:
            return {"kind": kind, "m": m, "p0": p0, "window": 512, "slots": 1024, "q_heads": qh, "kv_heads": kvh}
        return {"kind": kind, "m": m, "p0": p0, "window": 0, "slots": p0 + m + rng.randrange(64), "q_heads": qh,
                "kv_heads": kvh}
    if kind == "prompt":
        return {"kind": kind, "n": _log(rng, 16, 1024)}
    return {"kind": kind, "n": _log(rng, 6, 95)}


# ---- inputs: made from the seed alone, in the formats a model file holds -------------------------------------------

def _sub(seed, k):
    return (seed * 1000003 + 7919 * k + 1) & 0xFFFFFFFFFFFF


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _q40(seed, k, rows, cols):
    from e4b import formats
    return formats.synth_q40(_sub(seed, k), rows, cols, 0.02)


def _normal(seed, k, *shape, std=1.0):
    from e4b import formats
    return formats.synth_normal(_sub(seed, k), int(np.prod(shape)), 0.0, std).reshape(shape)


def _uniform(seed, k, n):
    return np.random.default_rng(_sub(seed, k)).uniform(0.5, 1.5, n).astype(np.float32)


def _moe_tensors(c, seed):
    H, E, FF, FD = c["hidden"], c["experts"], c["ff"], c["dense"]
    t = {"ffn_norm": _uniform(seed, 20, H), "router_scale": _uniform(seed, 21, H), "pre_ffw2": _uniform(seed, 22, H),
         "post_ffw1": _uniform(seed, 23, H), "post_ffw2": _uniform(seed, 24, H), "post_ffw": _uniform(seed, 25, H),
         "pes": _uniform(seed, 26, E), "router_w": _normal(seed, 27, E, H, std=0.02),
         "dense_gate": _q40(seed, 1, FD, H), "dense_up": _q40(seed, 2, FD, H), "dense_down": _q40(seed, 3, H, FD),
         "exp_gate_up": _q40(seed, 4, E * 2 * FF, H), "exp_down": _q40(seed, 5, E * H, FF)}
    return t, _normal(seed, 6, c.get("m", 1), H)


def _attn_inputs(c, seed):
    """Raw projections and caches as a running model holds them: normed keys, unit-rms values."""
    if c["kind"] == "attn_decode":
        qh, kvh = 8, 2
        qkv = _normal(seed, 30, (qh + 2 * kvh) * HEAD_DIM)
    else:
        qh, kvh = c["q_heads"], c["kv_heads"]
        qkv = _normal(seed, 30, c["m"], qh, HEAD_DIM)
    k = _normal(seed, 31, kvh, c["slots"], HEAD_DIM, std=0.25).astype(np.float16)
    v = _normal(seed, 32, kvh, c["slots"], HEAD_DIM).astype(np.float16)
    return qkv, k, v, _uniform(seed, 33, HEAD_DIM), 0.25 * _uniform(seed, 34, HEAD_DIM)


def _engine_model(seed):
    from e4b.model import E4BConfig, norm_weights_random, synth_tensors
    cfg = E4BConfig(layers=LAYERS, max_seq=MAX_SEQ)
    return cfg, norm_weights_random(synth_tensors(cfg, _sub(seed, 40)), _sub(seed, 41))


def _ids(c, seed, vocab):
    return np.random.default_rng(_sub(seed, 42)).integers(0, vocab, c["n"]).astype(np.uint32)


def prepare(case, seed):
    from e4b.kernels import MoeLayer, Q40Matrix, Q6KMatrix, rope_inv_freq
    c, kind = case, case["kind"]
    empty = lambda *s, dtype=torch.float32: torch.empty(*s, dtype=dtype, device="cuda")  # noqa: E731
    s = {"c": c}
    if kind == "gemv":
        x = _normal(seed, 2, c["cols"])
        s.update(w=Q40Matrix(_q40(seed, 1, c["rows"], c["cols"]), c["rows"], c["cols"]),
                 x=_gpu(x.astype(np.float16) if c["f16"] else x), y=empty(c["rows"]))
    elif kind == "lmhead":
        from e4b import formats
        w = formats.synth_q6k(_sub(seed, 1), c["rows"], c["cols"], 1e-3)
        s.update(w=Q6KMatrix(w, c["rows"], c["cols"]), x=_gpu(_normal(seed, 2, c["cols"])), y=empty(c["rows"]),
                 amax=empty(2, dtype=torch.int32))
    elif kind == "attn_decode":
        qkv, k, v, qw, kw = _attn_inputs(c, seed)
        theta = 1e4 if c["window"] else 1e6
        s.update(qkv=_gpu(qkv), k=_gpu(k), v=_gpu(v), qw=_gpu(qw), kw=_gpu(kw),
                 inv=_gpu(rope_inv_freq(theta, HEAD_DIM, HEAD_DIM // 2)), out=empty(8, HEAD_DIM, dtype=torch.float16))
    elif kind in ("moe", "moe_prefill"):
        t, h = _moe_tensors(c, seed)
        m = c.get("m", 1)
        s.update(w=MoeLayer(c["hidden"], c["experts"], c["ff"], c["dense"], t, EPS), h=_gpu(h),
                 h_out=empty(m, c["hidden"]), idx=empty(m, TOP_K, dtype=torch.int32), wts=empty(m, TOP_K),
                 dense=empty(m, c["hidden"]), moe=empty(m, c["hidden"]))
    elif kind == "gemm":
        s.update(w=Q40Matrix(_q40(seed, 1, c["rows"], c["cols"]), c["rows"], c["cols"]),
                 x=_gpu(_normal(seed, 2, c["m"], c["cols"]).astype(np.float16)), y=empty(c["m"], c["rows"]))
    elif kind == "geglu":
        s.update(w=Q40Matrix(_q40(seed, 1, 2 * c["ff"], c["cols"]), 2 * c["ff"], c["cols"]),
                 x=_gpu(_normal(seed, 2, c["m"], c["cols"]).astype(np.float16)),
                 y=empty(c["m"], c["ff"], dtype=torch.float16))
    elif kind == "attn_prefill":
        q, k, v, _, _ = _attn_inputs(c, seed)
        s.update(q=_gpu(q), k=_gpu(k), v=_gpu(v), out=empty(c["m"], c["q_heads"] * HEAD_DIM, dtype=torch.float16))
    else:
        from e4b.engine import Engine
        cfg, tensors = _engine_model(seed)
        s.update(eng=Engine(cfg, tensors), ids=_ids(c, seed, cfg.vocab))
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------

def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    from e4b._lib import DT_F16, DT_F32, check, lib
    s, c = state, state["c"]
    kind = c["kind"]
    if kind == "gemv":
        s["w"].gemv_dev(s["x"].data_ptr(), DT_F16 if c["f16"] else DT_F32, s["y"].data_ptr())
        return s["y"]
    if kind == "lmhead":
        s["w"].gemv_argmax_dev(s["x"].data_ptr(), SOFTCAP, s["y"].data_ptr(), s["amax"].data_ptr())
        return {"logits": s["y"], "index": s["amax"][:1], "max": s["amax"][1:].view(torch.float32)}
    if kind == "attn_decode":
        check(lib.e4b_k_attn_decode(_p(s["qkv"]), _p(s["qw"]), _p(s["kw"]), _p(s["inv"]), HEAD_DIM // 2, _p(s["k"]),
                                    _p(s["v"]), 8, 2, HEAD_DIM, c["slots"], c["window"], c["pos"],
                                    ctypes.c_float(EPS), 0, _p(s["out"]), None), "e4b_k_attn_decode")
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    if kind == "moe":
        check(lib.e4b_k_moe_layer(ctypes.byref(s["w"].w), _p(s["h"]), _p(s["h_out"]), _p(s["idx"]), _p(s["wts"]),
                                  _p(s["dense"]), _p(s["moe"]), None), "e4b_k_moe_layer")
        return {n: s[n] for n in ("h_out", "idx", "wts", "dense", "moe")}
    if kind == "moe_prefill":
        check(lib.e4b_k_moe_prefill(ctypes.byref(s["w"].w), _p(s["h"]), c["m"], _p(s["h_out"]), _p(s["idx"]),
                                    _p(s["wts"]), _p(s["dense"]), _p(s["moe"]), None), "e4b_k_moe_prefill")
        return {n: s[n] for n in ("h_out", "idx", "wts", "dense", "moe")}
    if kind == "gemm":
        s["w"].gemm_dev(s["x"].data_ptr(), c["m"], s["y"].data_ptr())
        return s["y"]
    if kind == "geglu":
        s["w"].gemm_geglu_dev(s["x"].data_ptr(), c["m"], s["y"].data_ptr())
        return s["y"]
    if kind == "attn_prefill":
        check(lib.e4b_k_attn_prefill(_p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["out"]), c["m"], c["q_heads"],
                                     c["kv_heads"], c["slots"], c["window"], c["p0"], None), "e4b_k_attn_prefill")
        return s["out"]
    eng = s["eng"]
    (eng.prefill if kind == "prompt" else eng.prefill_steps)(s["ids"])
    return {"logits": eng.read_logits(), "hidden": eng.read_hidden()} if kind == "steps" else eng.read_logits()


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _b40(rows, cols):
    return rows * cols // 32 * 18


def _keys(pos, window):
    return min(pos + 1, window) if window else pos + 1


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        r, k = c["rows"], c["cols"]
        return {"bytes": _b40(r, k) + k * (2 if c["f16"] else 4) + 4 * r, "flops": 2 * r * k}
    if kind == "lmhead":
        r, k = c["rows"], c["cols"]
        return {"bytes": r * (k // 256) * 210 + 4 * k + 4 * r + 8, "flops": 2 * r * k}
    if kind == "attn_decode":
        n = _keys(c["pos"], c["window"])
        return {"bytes": n * 2 * 2 * HEAD_DIM * 2 + 12 * HEAD_DIM * 4 + 8 * HEAD_DIM * 2 + 2 * 2 * HEAD_DIM * 2,
                "flops": 4 * n * 8 * HEAD_DIM}
    if kind in ("moe", "moe_prefill"):
        H, E, FF, FD, m = c["hidden"], c["experts"], c["ff"], c["dense"], c.get("m", 1)
        used = E * (1 - (1 - TOP_K / E) ** m)  # experts that m tokens reach, as if they chose evenly
        b = E * H * 4 + used * (_b40(2 * FF, H) + _b40(H, FF)) + _b40(2 * FD, H) + _b40(H, FD)
        return {"bytes": b + m * (4 * H * 4 + 64) + 6 * H * 4 + 4 * E,
                "flops": 2 * m * (E * H + 3 * H * (TOP_K * FF + FD))}
    if kind == "gemm":
        r, k, m = c["rows"], c["cols"], c["m"]
        return {"bytes": _b40(r, k) + 2 * m * k + 4 * m * r, "flops": 2 * m * r * k}
    if kind == "geglu":
        f, k, m = c["ff"], c["cols"], c["m"]
        return {"bytes": _b40(2 * f, k) + 2 * m * k + 2 * m * f, "flops": 4 * m * f * k}
    if kind == "attn_prefill":
        m, qh, kvh = c["m"], c["q_heads"], c["kv_heads"]
        pairs = sum(_keys(c["p0"] + i, c["window"]) for i in range(m))
        keys = min(c["p0"] + m, c["window"] + m - 1) if c["window"] else c["p0"] + m
        return {"bytes": keys * kvh * HEAD_DIM * 4 + m * qh * HEAD_DIM * 6, "flops": 4 * pairs * qh * HEAD_DIM}
    H, F, QH, KVH, PD, V, n = 2048, 16384, 8, 2, 256, 262144, c["n"]
    mats = LAYERS * ((QH + 2 * KVH) * HEAD_DIM * H + QH * HEAD_DIM * H + 3 * F * H + 2 * PD * H) + LAYERS * PD * H
    weights, head = mats // 32 * 18, V * H // 256 * 210
    rows = n * (H // 256 + LAYERS) * 210  # embedding and per-layer embedding rows
    kv_row = 2 * KVH * HEAD_DIM * 2
    live = sum(_keys(i, 0 if layer % 5 == 4 else 512) for layer in range(LAYERS) for i in range(n))
    flops = 2 * n * mats + 4 * live * QH * HEAD_DIM
    if kind == "prompt":
        return {"bytes": weights + head + rows + LAYERS * n * kv_row + 4 * V, "flops": flops + 2 * V * H}
    return {"bytes": n * (weights + head + 4 * V) + rows + live * kv_row, "flops": flops + 2 * n * V * H}


def tolerance(case):
    """About four times the distance from the 64-bit result that is measured (in brackets)."""
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1.5e-5}                  # f32 sums whose offset of 8 is taken out at the end (3.7e-6)
    if kind == "lmhead":
        return {"rel": 1e-5}                    # f32 activations as two 16-bit halves (2.3e-6)
    if kind == "gemm":
        return {"rel": 2e-6}                    # f32 sums of exact products, in another order (4.1e-7)
    if kind in ("geglu", "attn_decode", "attn_prefill"):
        return {"rel": 8e-4}                    # 16-bit results (2.1e-4)
    if kind in ("moe", "moe_prefill"):
        return {"rel": 3e-4, "differ": 0.002}   # 16-bit values between the matrices (7e-5); expert picks that tie
    return {"rel": 1e-3}                        # 16-bit roundings that flip in one layer travel on (2e-4)


# ---- the same in 64 bits, in plain torch ---------------------------------------------------------------------------

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev()).double()


def _r16(x):
    return x.to(torch.float16).double()


def _deq40(w, rows, cols):
    """q4_0 blocks (f16 scale, 16 bytes: elements 0-15 in the low nibbles, 16-31 in the high ones)."""
    b = torch.from_numpy(np.ascontiguousarray(w).reshape(-1, 18)).to(_dev())
    d = b[:, :2].contiguous().view(torch.float16).double()
    q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
    return (q * d).reshape(rows, cols)


def _deq6k(w, cols):
    """Q6_K superblocks of 256 (128 bytes of low nibbles, 64 of high bit pairs, 16 int8 scales, f16 scale)."""
    b = torch.from_numpy(np.ascontiguousarray(w).reshape(-1, 210)).to(_dev())
    lo, hi = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
    low = torch.cat([lo & 15, lo >> 4], 2)                                     # [n][half][quarter][32]
    shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
    q = (low | (((hi >> shift) & 3) << 4)).double() - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(-1, 16, 1)
    d = b[:, 208:].contiguous().view(torch.float16).double().reshape(-1, 1, 1)
    return (q.reshape(-1, 16, 16) * sc * d).reshape(-1, cols)


def _rms(x):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt()


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh((math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)).clamp(-20, 20)))


def _rope(x, pos, theta):
    """NeoX rotation of pairs (p, p + 128); x [..., tokens, heads, 256], the angle in f32 as a model's tables hold it."""
    half = HEAD_DIM // 2
    inv = (theta ** (-2.0 * torch.arange(half, dtype=torch.float64) / HEAD_DIM)).float().to(x.device)
    a = (pos.float()[:, None, None] * inv).double()
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def _attend(q, k, v, qpos, kpos, window):
    """q [m][qh][256], k and v [n][kvh][256]: causal softmax attention, scores not scaled."""
    g = q.shape[1] // k.shape[1]
    live = kpos[None, :] <= qpos[:, None]
    if window:
        live &= kpos[None, :] > qpos[:, None] - window
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // g].T).masked_fill(~live, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // g]
    return out


def _exact_moe(c, seed):
    t, hin = _moe_tensors(c, seed)
    H, E, FF, FD = c["hidden"], c["experts"], c["ff"], c["dense"]
    h = _f64(hin)
    f = {n: _f64(t[n]) for n in t if t[n].dtype == np.float32}
    n = _rms(h)
    xd, xm = _r16(n * f["ffn_norm"]), _r16(n * f["pre_ffw2"])
    scores = (n * f["router_scale"] / math.sqrt(H)) @ f["router_w"].T
    p = torch.softmax(scores, -1)
    top = torch.sort(p, dim=-1, descending=True, stable=True)[1][:, :TOP_K]
    pk = p.gather(1, top)
    wts = pk / pk.sum(-1, keepdim=True) * f["pes"][top]
    g = _gelu(xd @ _deq40(t["dense_gate"], FD, H).T) * (xd @ _deq40(t["dense_up"], FD, H).T)
    dense = _r16(g) @ _deq40(t["dense_down"], H, FD).T
    moe = torch.zeros_like(h)
    gu = np.ascontiguousarray(t["exp_gate_up"]).reshape(E, -1)
    dn = np.ascontiguousarray(t["exp_down"]).reshape(E, -1)
    for e in range(E):
        tok, slot = (top == e).nonzero(as_tuple=True)
        if tok.numel():
            y = xm[tok] @ _deq40(gu[e], 2 * FF, H).T
            y = _r16(_gelu(y[:, :FF]) * y[:, FF:]) @ _deq40(dn[e], H, FF).T
            moe.index_add_(0, tok, y * wts[tok, slot, None])
    comb = _rms(dense) * f["post_ffw1"] + _rms(moe) * f["post_ffw2"]
    return {"h_out": h + _rms(comb) * f["post_ffw"], "idx": None, "wts": wts, "dense": dense, "moe": moe}


def _exact_engine(c, seed):
    cfg, t = _engine_model(seed)
    ids = torch.from_numpy(_ids(c, seed, cfg.vocab).astype(np.int64))
    H, F, PD, V, QH, KVH, D = cfg.hidden, cfg.ffn, cfg.ple_dim, cfg.vocab, cfg.q_heads, cfg.kv_heads, HEAD_DIM
    f32 = lambda n: _f64(t[n].data)  # noqa: E731
    q40 = lambda n, r, k: _deq40(t[n].data, r, k)  # noqa: E731

    def rows6(n, cols):
        return _deq6k(np.ascontiguousarray(t[n].data).reshape(V, -1)[ids.numpy()], cols)

    h = rows6("token_embd.weight", H) * math.sqrt(H)
    proj = (h @ q40("per_layer_model_proj.weight", LAYERS * PD, H).T / math.sqrt(H)).reshape(-1, LAYERS, PD)
    ple = _rms(proj) * f32("per_layer_proj_norm.weight")
    ple = (ple + rows6("per_layer_token_embd.weight", LAYERS * PD).reshape(-1, LAYERS, PD) * math.sqrt(PD)) / math.sqrt(2)
    pos = torch.arange(c["n"], device=h.device)
    for i in range(LAYERS):
        b, glob = f"blk.{i}.", bool(cfg.layer_global[i])
        theta = cfg.theta_global if glob else cfg.theta_local
        x = _r16(_rms(h) * f32(b + "attn_norm.weight"))
        q = (x @ q40(b + "attn_q.weight", QH * D, H).T).reshape(-1, QH, D)
        k = (x @ q40(b + "attn_k.weight", KVH * D, H).T).reshape(-1, KVH, D)
        v = (x @ q40(b + "attn_v.weight", KVH * D, H).T).reshape(-1, KVH, D)
        q = _rope(_rms(q) * f32(b + "attn_q_norm.weight"), pos, theta)
        k = _r16(_rope(_rms(k) * f32(b + "attn_k_norm.weight"), pos, theta))
        a = _attend(q, k, _r16(_rms(v)), pos, pos, 0 if glob else cfg.window)
        o = _r16(a.reshape(-1, QH * D)) @ q40(b + "attn_output.weight", H, QH * D).T
        h = h + _rms(o) * f32(b + "post_attention_norm.weight")
        x = _r16(_rms(h) * f32(b + "ffn_norm.weight"))
        g = _gelu(x @ q40(b + "ffn_gate.weight", F, H).T) * (x @ q40(b + "ffn_up.weight", F, H).T)
        h = h + _rms(_r16(g) @ q40(b + "ffn_down.weight", H, F).T) * f32(b + "post_ffw_norm.weight")
        g = _r16(_gelu(_r16(h) @ q40(b + "inp_gate.weight", PD, H).T) * ple[:, i])
        h = h + _rms(g @ q40(b + "proj.weight", H, PD).T) * f32(b + "post_norm.weight")
        h = h * f32(b + "layer_output_scale.weight")
    x = _rms(h[-1]) * f32("output_norm.weight")
    head = np.ascontiguousarray(t["token_embd.weight"].data).reshape(V, -1)
    logits = torch.cat([_deq6k(head[r:r + 32768], H) @ x for r in range(0, V, 32768)])
    logits = SOFTCAP * torch.tanh(logits / SOFTCAP)
    return {"logits": logits, "hidden": h[-1]} if c["kind"] == "steps" else logits


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        x = _normal(seed, 2, c["cols"])
        return _deq40(_q40(seed, 1, c["rows"], c["cols"]), c["rows"], c["cols"]) @ _f64(
            x.astype(np.float16) if c["f16"] else x)
    if kind == "lmhead":
        from e4b import formats
        x = _f64(_normal(seed, 2, c["cols"]))
        w = formats.synth_q6k(_sub(seed, 1), c["rows"], c["cols"], 1e-3).reshape(c["rows"], -1)
        y = torch.cat([_deq6k(w[r:r + 32768], c["cols"]) @ x for r in range(0, c["rows"], 32768)])
        y = SOFTCAP * torch.tanh(y / SOFTCAP)
        return {"logits": y, "index": None, "max": y.max().reshape(1)}
    if kind == "attn_decode":
        qkv, k, v, qw, kw = _attn_inputs(c, seed)
        pos, theta = c["pos"], 1e4 if c["window"] else 1e6
        z = _f64(qkv).reshape(1, 12, HEAD_DIM)
        at = torch.tensor([pos], device=z.device)
        q = _rope(_rms(z[:, :8]) * _f64(qw), at, theta)
        kc, vc = _f64(k).transpose(0, 1).clone(), _f64(v).transpose(0, 1).clone()
        kc[pos % c["slots"]] = _r16(_rope(_rms(z[:, 8:10]) * _f64(kw), at, theta))[0]
        vc[pos % c["slots"]] = _r16(_rms(z[:, 10:]))[0]
        kpos = torch.arange(max(0, pos - c["window"] + 1) if c["window"] else 0, pos + 1, device=z.device)
        out = _attend(q, kc[kpos % c["slots"]], vc[kpos % c["slots"]], at, kpos, c["window"])[0]
        return {"out": out, "k": kc.transpose(0, 1).contiguous(), "v": vc.transpose(0, 1).contiguous()}
    if kind in ("moe", "moe_prefill"):
        return _exact_moe(c, seed)
    if kind == "gemm":
        x = _f64(_normal(seed, 2, c["m"], c["cols"]).astype(np.float16))
        return x @ _deq40(_q40(seed, 1, c["rows"], c["cols"]), c["rows"], c["cols"]).T
    if kind == "geglu":
        x = _f64(_normal(seed, 2, c["m"], c["cols"]).astype(np.float16))
        y = x @ _deq40(_q40(seed, 1, 2 * c["ff"], c["cols"]), 2 * c["ff"], c["cols"]).T
        return _gelu(y[:, :c["ff"]]) * y[:, c["ff"]:]
    if kind == "attn_prefill":
        q, k, v, _, _ = _attn_inputs(c, seed)
        p0, m, window = c["p0"], c["m"], c["window"]
        q = _f64(q)
        kpos = torch.arange(max(0, p0 - window + 1) if window else 0, p0 + m, device=q.device)
        kc, vc = _f64(k).transpose(0, 1)[kpos % c["slots"]], _f64(v).transpose(0, 1)[kpos % c["slots"]]
        out = _attend(q, kc, vc, torch.arange(p0, p0 + m, device=q.device), kpos, window)
        return out.reshape(m, -1)
    return _exact_engine(c, seed)
