"""Performance cases: the work a program built on this library has it do.

Five kinds of call, each through the public entry points of g4hip:

  host_matvec  FloatTensor.matmul on host arrays, the drop-in boundary of the
               reference: one synchronous call per matrix (latency).
  decode       one token through several layers with its activations in device
               memory: norm + projections, KV-cache attention (one global layer
               in six, the others with a sliding window), output projection,
               post-norm and the dense FFN block.  Recorded once as a HIP graph
               and replayed per token, as a decode loop does.
  lm_head      final norm, logits over the vocabulary, soft-cap and arg-max.
  batch        several tokens against one matrix (matmul_batch_dev): a few
               sequences decoded together (recorded as a graph over the matrices
               of a step) or a prompt's tokens (called eagerly).
  moe          routed Q4_K experts (moe_routed_dev): single decode tokens, a
               small batch, a prompt.

Weights are random GGUF blocks whose values are centred on zero, as trained
weights are, and scaled so that a row's sum has the activations' size.  States
hold enough distinct weights that a pass streams them from memory, not from a
cache that the previous pass filled.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "gemma4.kt_amd"))

import g4hip  # noqa: E402

_T = {"F32": 0, "F16": 1, "Q4_0": 2, "Q8_0": 8, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "BF16": 30}
_BLOCK = {"F32": (1, 4), "F16": (1, 2), "BF16": (1, 2), "Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144),
          "Q5_K": (256, 176), "Q6_K": (256, 210)}
_EPS = 1e-6
_CAP = 30.0

# the widths of the configured decode layer and of its attention
_DIM, _HIDDEN, _HEADS, _KV_HEADS, _HEAD = 2048, 8192, 16, 8, 256


def listed():
    return [
        # one matrix of the smallest configured size on host arrays: what a host
        # program that only swaps its tensor class calls
        {"name": "host_matvec_q8_0", "kind": "host_matvec", "type": "Q8_0", "rows": 2048, "cols": 2048},
        # a token of a chat with about a thousand tokens of context, 4-bit weights
        {"name": "decode_q4_0_ctx1k", "kind": "decode", "type": "Q4_0", "down_type": "Q4_0", "layers": 6, "pos": 1000,
         "window": 512},
        # a token deep in a long context, the mixed K-quant file (Q4_K with Q6_K
        # for the down projections and values)
        {"name": "decode_q4_k_ctx8k", "kind": "decode", "type": "Q4_K", "down_type": "Q6_K", "layers": 6, "pos": 8191,
         "window": 1024},
        # the vocabulary projection of every generated token
        {"name": "lm_head_q8_0", "kind": "lm_head", "type": "Q8_0", "rows": 262144, "cols": 2048},
        # eight sequences decoded together
        {"name": "batch8_q4_k", "kind": "batch", "type": "Q4_K", "rows": 8192, "cols": 2048, "m": 8, "layers": 16,
         "captured": True},
        # sixty-four sequences decoded together
        {"name": "batch64_q4_k", "kind": "batch", "type": "Q4_K", "rows": 8192, "cols": 2048, "m": 64, "layers": 12,
         "captured": True},
        # sequences decoded together on the 8-bit file
        {"name": "batch19_q8_0", "kind": "batch", "type": "Q8_0", "rows": 8192, "cols": 2048, "m": 19, "layers": 8,
         "captured": True},
        # a prompt chunk on K-quant weights
        {"name": "prompt512_q4_k", "kind": "batch", "type": "Q4_K", "rows": 8192, "cols": 2048, "m": 512, "layers": 2,
         "captured": False},
        # a short prompt of no round length through wide down projections
        {"name": "prompt201_q4_0", "kind": "batch", "type": "Q4_0", "rows": 2048, "cols": 8192, "m": 201, "layers": 2,
         "captured": False},
        # eight tokens decoded one after the other through routed experts
        {"name": "moe_token", "kind": "moe", "tokens": 1, "calls": 8, "experts": 128, "dim": 2048, "ff": 1408, "k": 8},
        # sixteen sequences decoded together through routed experts
        {"name": "moe_16", "kind": "moe", "tokens": 16, "calls": 1, "experts": 128, "dim": 2048, "ff": 1408, "k": 8},
        # a prompt through routed experts
        {"name": "moe_prompt_200", "kind": "moe", "tokens": 200, "calls": 1, "experts": 128, "dim": 2048, "ff": 1408,
         "k": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host_matvec", "decode", "lm_head", "batch", "batch", "batch", "batch", "moe", "moe"])
    if kind == "host_matvec":
        t = rng.choice(["Q8_0", "Q4_0", "Q4_K", "Q6_K"])
        return {"kind": kind, "type": t, "rows": _log(rng, 256, 8192), "cols": 256 * rng.randint(2, 16)}
    if kind == "decode":
        t, d = rng.choice([("Q4_0", "Q4_0"), ("Q8_0", "Q8_0"), ("Q4_K", "Q6_K"), ("Q5_K", "Q6_K")])
        return {"kind": kind, "type": t, "down_type": d, "layers": rng.randint(4, 6) if t != "Q8_0" else 3,
                "pos": _log(rng, 30, 8191), "window": rng.choice([512, 1024])}
    if kind == "lm_head":
        t = rng.choice(["Q8_0", "Q6_K", "Q4_K"])
        return {"kind": kind, "type": t, "rows": _log(rng, 30000, 262144), "cols": 256 * rng.randint(4, 8)}
    if kind == "batch":
        t = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q4_0", "Q5_K", "Q6_K", "F16", "BF16"])
        small = rng.random() < 0.5
        m = _log(rng, 2, 64) if small else _log(rng, 65, 512)
        cols = (32 * rng.randint(16, 128) if t in ("Q8_0", "Q4_0") and rng.random() < 0.5
                else 256 * rng.randint(2, 32))
        rows = _log(rng, 1000, 8192)
        while rows * cols > 8192 * 2048:
            rows = max(500, rows // 2 + 1)
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "m": m, "layers": 8 if small else 2,
                "captured": small}
    t = _log(rng, 1, 200)
    return {"kind": "moe", "tokens": t, "calls": 8 if t == 1 else 2 if t < 16 else 1,
            "experts": rng.choice([32, 64, 128]), "dim": rng.choice([1024, 1536, 2048]),
            "ff": rng.choice([704, 768, 1024, 1408]), "k": rng.choice([2, 4, 6, 8])}


# ------------------------------------------------------------------ inputs ---

def _bytes(gen, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _half(v):
    """float -> its two fp16 bytes, [n, 2]."""
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(-1, 2)


def _raw(gen, typ, rows, cols):
    """rows x cols random weights of a GGUF type as their raw blocks (uint8, on the GPU)."""
    n = rows * cols
    bs, ts = _BLOCK[typ]
    s = 1.0 / math.sqrt(cols)  # a weight's size: a row's sum then has the activations' size
    if typ in ("F32", "F16", "BF16"):
        v = torch.randn(n, device="cuda", generator=gen) * s
        return v.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[typ]).view(torch.uint8)
    nb = n // bs
    out = _bytes(gen, nb, ts)
    d = torch.rand(nb, device="cuda", generator=gen) + 0.5
    if typ == "Q8_0":
        out[:, 0:2] = _half(d * (s / 74.0))
    elif typ == "Q4_0":
        out[:, 0:2] = _half(d * (s / 4.6))
    elif typ == "Q6_K":
        sc = torch.randint(32, 128, (nb, 16), device="cuda", generator=gen, dtype=torch.int16)
        neg = torch.rand(nb, 16, device="cuda", generator=gen) < 0.5
        out[:, 192:208] = (torch.where(neg, -sc, sc) & 255).to(torch.uint8)
        out[:, 208:210] = _half(d * (s / (18.0 * 85.0)))
    else:  # Q4_K, Q5_K: d * sc * q - dmin * m, the mins at the middle of the scale's range
        mid = 7.5 if typ == "Q4_K" else 15.5
        d = d * (s / (mid * 0.62 * 48.0))
        out[:, 0:2] = _half(d)
        out[:, 2:4] = _half(d * mid)
        sc = torch.randint(32, 64, (nb, 8), device="cuda", generator=gen, dtype=torch.int16)
        m = (sc + torch.randint(-2, 3, (nb, 8), device="cuda", generator=gen, dtype=torch.int16)).clamp(0, 63)
        out[:, 4:8] = ((sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        out[:, 8:12] = ((m[:, :4] & 63) | ((m[:, 4:] >> 4) << 6)).to(torch.uint8)
        out[:, 12:16] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
    return out.reshape(-1)


def _normal(gen, *shape, scale=1.0):
    return torch.randn(*shape, device="cuda", generator=gen) * scale


def _norm_weight(gen, n, scale=1.0):
    return scale * (1.0 + 0.25 * torch.randn(n, device="cuda", generator=gen))


def _inputs(case, seed):
    """Every input of a case as GPU tensors, from the seed alone (weights as raw blocks)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "host_matvec":
        return {"w": _raw(gen, case["type"], case["rows"], case["cols"]), "x": _normal(gen, case["cols"])}
    if kind == "lm_head":
        return {"w": _raw(gen, case["type"], case["rows"], case["cols"]),
                "norm": _norm_weight(gen, case["cols"], 3.0), "x": _normal(gen, case["cols"], scale=4.0)}
    if kind == "batch":
        return {"w": [_raw(gen, case["type"], case["rows"], case["cols"]) for _ in range(case["layers"])],
                "x": [_normal(gen, case["m"], case["cols"]) for _ in range(case["layers"])]}
    if kind == "moe":
        E, dim, ff = case["experts"], case["dim"], case["ff"]
        return {"gate_up": _raw(gen, "Q4_K", E * 2 * ff, dim), "down": _raw(gen, "Q4_K", E * dim, ff),
                "logits": [_normal(gen, case["tokens"], E) for _ in range(case["calls"])],
                "x": [_normal(gen, case["tokens"], dim) for _ in range(case["calls"])]}
    q, kv, t, n = _HEADS * _HEAD, _KV_HEADS * _HEAD, case["type"], case["pos"] + 1
    layers = []
    for _ in range(case["layers"]):
        layers.append({
            "wq": (t, q, _DIM, _raw(gen, t, q, _DIM)), "wk": (t, kv, _DIM, _raw(gen, t, kv, _DIM)),
            "wv": (case["down_type"], kv, _DIM, _raw(gen, case["down_type"], kv, _DIM)),
            "wo": (t, _DIM, q, _raw(gen, t, _DIM, q)),
            "gate": (t, _HIDDEN, _DIM, _raw(gen, t, _HIDDEN, _DIM)),
            "up": (t, _HIDDEN, _DIM, _raw(gen, t, _HIDDEN, _DIM)),
            "down": (case["down_type"], _DIM, _HIDDEN, _raw(gen, case["down_type"], _DIM, _HIDDEN)),
            "n_att": _norm_weight(gen, _DIM), "n_att_post": _norm_weight(gen, _DIM),
            "n_ffn": _norm_weight(gen, _DIM), "n_ffn_post": _norm_weight(gen, _DIM),
            # per-head norms: queries and keys small enough that a softmax over
            # many positions is neither flat nor one position
            "n_q": _norm_weight(gen, _HEAD, 0.35), "n_k": _norm_weight(gen, _HEAD, 0.35),
            "kc": _normal(gen, n, kv, scale=0.35), "vc": _normal(gen, n, kv)})
    return {"layers": layers, "emb": _normal(gen, _DIM, scale=1.0 / math.sqrt(_DIM))}


# ------------------------------------------------------------------- state ---

_ctx = None
_stream = None


def _context():
    """The program's one context, with its scratch reserved up front (graphs are
    recorded over it)."""
    global _ctx, _stream
    if _ctx is None:
        _ctx = g4hip.Context(0)
        _ctx.reserve(256 << 20)
        _stream = torch.cuda.Stream()
    return _ctx


def _weight(ctx, typ, raw, n):
    torch.cuda.synchronize()
    return g4hip.FloatTensorFactory.create(ctx, _T[typ], raw.cpu().numpy(), n)


def _norm(ctx, v):
    return _weight(ctx, "F32", v.view(torch.uint8), v.numel())


def _recorded(ctx, step):
    """`step` as a HIP graph, after one eager run of it."""
    step()
    ctx.sync()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=_stream):
        ctx.set_stream(_stream.cuda_stream)
        step()
    ctx.set_stream(None)
    torch.cuda.synchronize()
    return g


def prepare(case, seed):
    ctx = _context()
    d = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case, "ctx": ctx, "graph": None}
    if kind == "host_matvec":
        s["w"] = _weight(ctx, case["type"], d["w"], case["rows"] * case["cols"])
        s["x"] = d["x"].cpu().numpy()
        s["y"] = np.empty(case["rows"], np.float32)
        return s
    if kind == "lm_head":
        s["w"] = _weight(ctx, case["type"], d["w"], case["rows"] * case["cols"])
        s["norm"] = _norm(ctx, d["norm"])
        s["x"] = d["x"]
        s["logits"] = torch.empty(case["rows"], device="cuda")
        s["index"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        return s
    if kind == "batch":
        s["w"] = [_weight(ctx, case["type"], w, case["rows"] * case["cols"]) for w in d["w"]]
        s["x"] = d["x"]
        s["y"] = [torch.empty(case["m"], case["rows"], device="cuda") for _ in d["w"]]
        if case["captured"]:
            s["graph"] = _recorded(ctx, lambda: _batch(s))
        return s
    if kind == "moe":
        E, dim, ff, t, k = case["experts"], case["dim"], case["ff"], case["tokens"], case["k"]
        s["gate_up"] = _weight(ctx, "Q4_K", d["gate_up"], E * 2 * ff * dim)
        s["down"] = _weight(ctx, "Q4_K", d["down"], E * dim * ff)
        s["logits"], s["x"] = d["logits"], d["x"]
        s["ids"] = [torch.zeros(t, k, dtype=torch.int32, device="cuda") for _ in d["x"]]
        s["gates"] = [torch.zeros(t, k, device="cuda") for _ in d["x"]]
        s["y"] = [torch.empty(t, dim, device="cuda") for _ in d["x"]]
        if case["calls"] > 1:
            s["graph"] = _recorded(ctx, lambda: _moe(s))
        return s
    s["emb"] = d["emb"]
    s["x"] = torch.empty(_DIM, device="cuda")
    s["xb"] = torch.empty(_DIM, device="cuda")
    s["q"] = torch.empty(_HEADS * _HEAD, device="cuda")
    s["att"] = torch.empty(_HEADS * _HEAD, device="cuda")
    s["layers"] = []
    for lay in d["layers"]:
        L = {}
        for name, v in lay.items():
            if name.startswith("w") or name in ("gate", "up", "down"):
                L[name] = _weight(ctx, v[0], v[3], v[1] * v[2])
            elif name.startswith("n_"):
                L[name] = _norm(ctx, v)
            else:
                L[name] = v
        L["k_row"], L["v_row"] = L["kc"][case["pos"]], L["vc"][case["pos"]]
        s["layers"].append(L)
    s["graph"] = _recorded(ctx, lambda: _decode(s))
    return s


# --------------------------------------------------------------------- run ---

def _start(case, layer):
    """First attended position: one layer in six (the last) is global."""
    return 0 if layer % 6 == 5 else max(0, case["pos"] - case["window"] + 1)


def _batch(s):
    c = s["case"]
    for w, x, y in zip(s["w"], s["x"], s["y"]):
        w.matmul_batch_dev(x, c["m"], y, c["rows"], c["cols"])


def _moe(s):
    c = s["case"]
    for lg, x, ids, gates, y in zip(s["logits"], s["x"], s["ids"], s["gates"], s["y"]):
        g4hip.moe_routed_dev(s["ctx"], s["gate_up"], s["down"], x, c["tokens"], c["dim"], c["ff"], lg, c["experts"],
                             c["k"], True, ids, gates, y)


def _decode(s):
    c, ctx, x, xb, q, att = s["case"], s["ctx"], s["x"], s["xb"], s["q"], s["att"]
    nq, nkv = _HEADS * _HEAD, _KV_HEADS * _HEAD
    torch.mul(s["emb"], math.sqrt(_DIM), out=x)  # the embedding row, scaled
    for i, L in enumerate(s["layers"]):
        g4hip.matmul_norm_dev(ctx, L["wq"], L["n_att"], x, q, nq, _DIM, _EPS)
        g4hip.matmul_norm_dev(ctx, L["wk"], L["n_att"], x, L["k_row"], nkv, _DIM, _EPS)
        g4hip.matmul_norm_dev(ctx, L["wv"], L["n_att"], x, L["v_row"], nkv, _DIM, _EPS)
        g4hip.rmsnorm_dev(ctx, L["n_q"], q, q, _HEADS, _HEAD, _EPS, g4hip.NORM_WEIGHT_FIRST)
        g4hip.rmsnorm_dev(ctx, L["n_k"], L["k_row"], L["k_row"], _KV_HEADS, _HEAD, _EPS, g4hip.NORM_WEIGHT_FIRST)
        g4hip.rmsnorm_dev(ctx, None, L["v_row"], L["v_row"], _KV_HEADS, _HEAD, _EPS, g4hip.NORM_NO_WEIGHT)
        g4hip.attention_dev(ctx, q, L["kc"], L["vc"], att, _HEADS, _KV_HEADS, _HEAD, c["pos"], _start(c, i))
        L["wo"].matmul_dev(att, xb, _DIM, nq)
        g4hip.rmsnorm_add_dev(ctx, L["n_att_post"], xb, x, _DIM, _EPS)
        g4hip.ffn_block_dev(ctx, L["gate"], L["up"], L["down"], L["n_ffn"], L["n_ffn_post"], x, _DIM, _HIDDEN, _EPS)


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "host_matvec":
        s["w"].matmul(s["x"], s["y"], c["rows"], c["cols"])
        return s["y"]
    if kind == "lm_head":
        g4hip.lm_head_dev(s["ctx"], s["w"], s["norm"], s["x"], s["logits"], s["index"], c["rows"], c["cols"], _EPS,
                          _CAP)
        return [s["logits"], s["index"]]
    if kind == "decode":
        s["graph"].replay()
        return {"x": s["x"], "keys": [L["k_row"] for L in s["layers"]], "values": [L["v_row"] for L in s["layers"]]}
    if s["graph"] is not None:
        s["graph"].replay()
    elif kind == "batch":
        _batch(s)
    else:
        _moe(s)
    return s["y"] if kind == "batch" else {"y": s["y"], "gates": s["gates"], "ids": s["ids"]}


# ------------------------------------------------------------- accounting ---

def _nbytes(typ, n):
    bs, ts = _BLOCK[typ]
    return n // bs * ts


def work(case):
    kind = case["kind"]
    if kind in ("host_matvec", "lm_head"):
        n = case["rows"] * case["cols"]
        return {"bytes": _nbytes(case["type"], n) + 4 * (case["rows"] + case["cols"]), "flops": 2 * n}
    if kind == "batch":
        n, m = case["rows"] * case["cols"], case["m"]
        return {"bytes": case["layers"] * (_nbytes(case["type"], n) + 4 * m * (case["rows"] + case["cols"])),
                "flops": case["layers"] * 2 * m * n}
    if kind == "moe":
        per, E = 3 * case["ff"] * case["dim"], case["experts"]
        pairs = case["calls"] * case["tokens"] * case["k"]
        # the experts that uniform routing is expected to reach
        hit = E * (1 - (1 - case["k"] / E) ** (case["calls"] * case["tokens"]))
        return {"bytes": hit * _nbytes("Q4_K", per) + 4 * case["calls"] * case["tokens"] * (2 * case["dim"] + E),
                "flops": 2 * pairs * per}
    q, kv = _HEADS * _HEAD, _KV_HEADS * _HEAD
    n_t = _DIM * (2 * q + kv + 2 * _HIDDEN)
    n_d = _DIM * (kv + _HIDDEN)
    nbytes = case["layers"] * (_nbytes(case["type"], n_t) + _nbytes(case["down_type"], n_d))
    flops = case["layers"] * 2 * (n_t + n_d)
    for i in range(case["layers"]):
        pos = case["pos"] + 1 - _start(case, i)
        nbytes += 2 * 4 * pos * kv
        flops += 4 * pos * q
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # fp32 sums in another order: measured against 64 bits, 1e-7 to 5e-7 for one
    # product, 4e-7 to 7e-7 for the experts' two, and up to 2.4e-6 in decode, where a
    # layer's rounding travels through the attention's exponentials and the layers
    # that follow.  Indices and expert ids may differ only by ties.
    if case["kind"] == "decode":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] == "moe":
        return {"rel": 3e-6, "max": 1e-4, "differ": 1e-3}
    if case["kind"] == "lm_head":
        return {"rel": 2e-6, "max": 1e-4, "differ": 0.0}
    return {"rel": 2e-6, "max": 1e-4}


# ------------------------------------------------------------------- exact ---

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(typ, raw, rows, cols):
    """Raw blocks -> float64 [rows, cols]."""
    bs, ts = _BLOCK[typ]
    if typ in ("F32", "F16", "BF16"):
        v = raw.contiguous().view({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[typ])
        return v.double().reshape(rows, cols)
    b = raw.reshape(-1, ts)
    if typ == "Q8_0":
        v = _f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif typ == "Q4_0":
        q = b[:, 2:]
        v = _f16(b[:, :2]) * (torch.cat([q & 15, q >> 4], 1).double() - 8)
    elif typ == "Q6_K":
        ql, qh = b[:, :128].reshape(-1, 2, 64).short(), b[:, 128:192].reshape(-1, 2, 32).short()
        lo, hi = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([(lo & 15) | ((qh & 3) << 4), (hi & 15) | (((qh >> 2) & 3) << 4),
                         (lo >> 4) | (((qh >> 4) & 3) << 4), (hi >> 4) | (((qh >> 6) & 3) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = _f16(b[:, 208:210])[:, :, None] * sc[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)
    else:
        s = b[:, 4:16].short()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        if typ == "Q5_K":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8)[None, :, None]
            q = q + 16 * ((b[:, None, 16:48] >> bit) & 1).double()
        v = (_f16(b[:, :2]) * sc)[:, :, None] * q - (_f16(b[:, 2:4]) * m)[:, :, None]
    return v.reshape(rows, cols)


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))


def _rms(v):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + _EPS)


def _exact_decode(case, d):
    x = d["emb"].double() * math.sqrt(_DIM)
    keys, values = [], []

    def mul(w, v):
        return _dequant(w[0], w[3], w[1], w[2]) @ v

    for i, L in enumerate(d["layers"]):
        h = _rms(x) * L["n_att"].double()
        q = _rms(mul(L["wq"], h).reshape(_HEADS, _HEAD)) * L["n_q"].double()
        k = (_rms(mul(L["wk"], h).reshape(_KV_HEADS, _HEAD)) * L["n_k"].double()).reshape(-1)
        v = _rms(mul(L["wv"], h).reshape(_KV_HEADS, _HEAD)).reshape(-1)
        keys.append(k)
        values.append(v)
        at = _start(case, i)
        kc, vc = L["kc"][at:].double(), L["vc"][at:].double()
        kc[-1], vc[-1] = k, v
        out = []
        for head in range(_HEADS):
            cols = slice(head // (_HEADS // _KV_HEADS) * _HEAD, (head // (_HEADS // _KV_HEADS) + 1) * _HEAD)
            out.append(torch.softmax(kc[:, cols] @ q[head], 0) @ vc[:, cols])
        x = x + _rms(mul(L["wo"], torch.cat(out))) * L["n_att_post"].double()
        h = _rms(x) * L["n_ffn"].double()
        h = _gelu(mul(L["gate"], h)) * mul(L["up"], h)
        x = x + _rms(mul(L["down"], h)) * L["n_ffn_post"].double()
    return {"x": x, "keys": keys, "values": values}


def _exact_moe(case, d):
    E, dim, ff, k = case["experts"], case["dim"], case["ff"], case["k"]
    per_gu = _nbytes("Q4_K", 2 * ff * dim)
    per_dn = _nbytes("Q4_K", dim * ff)
    picks = []
    for lg in d["logits"]:
        p = torch.softmax(lg.double(), 1)
        w, ids = torch.topk(p, k, 1)
        picks.append((ids, w / w.sum(1, keepdim=True)))
    y = [torch.zeros(case["tokens"], dim, dtype=torch.float64, device="cuda") for _ in d["x"]]
    for e in range(E):
        hits = [(c, (ids == e).nonzero()) for c, (ids, _) in enumerate(picks)]
        if not any(len(at) for _, at in hits):
            continue
        gu = _dequant("Q4_K", d["gate_up"][e * per_gu:(e + 1) * per_gu], 2 * ff, dim)
        dn = _dequant("Q4_K", d["down"][e * per_dn:(e + 1) * per_dn], dim, ff)
        for c, at in hits:
            if len(at):
                r = d["x"][c][at[:, 0]].double() @ gu.T
                r = (_gelu(r[:, :ff]) * r[:, ff:]) @ dn.T
                y[c].index_add_(0, at[:, 0], r * picks[c][1][at[:, 0], at[:, 1]][:, None])
    return {"y": y, "gates": [w for _, w in picks], "ids": [i.int() for i, _ in picks]}


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "host_matvec":
        return (_dequant(case["type"], d["w"], case["rows"], case["cols"]) @ d["x"].double()).cpu().numpy()
    if kind == "lm_head":
        h = _rms(d["x"].double()) * d["norm"].double()
        per = _nbytes(case["type"], case["cols"])
        step = 16384
        v = torch.cat([_dequant(case["type"], d["w"][r * per:min(case["rows"], r + step) * per],
                                min(case["rows"], r + step) - r, case["cols"]) @ h
                       for r in range(0, case["rows"], step)])
        v = _CAP * torch.tanh(v / _CAP)
        return [v, v.argmax().int().reshape(1)]
    if kind == "batch":
        return [x.double() @ _dequant(case["type"], w, case["rows"], case["cols"]).T for w, x in zip(d["w"], d["x"])]
    if kind == "moe":
        return _exact_moe(case, d)
    return _exact_decode(case, d)
