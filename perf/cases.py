"""Performance cases: the work a program has this library do, through its public entry points.

A GGUF runtime calls the library in four ways: mat-vecs for each decoded token
(device pointers, or the host-buffer entry of the Java drop-in), GEMMs for a
batch of decoding sequences or the tokens of a prompt, and the routed MoE block
for both.  The listed cases are those calls at the sizes of 7B-class and
128-expert models; draw() gives others of the same ranges: ragged row counts,
odd batch sizes, every weight type, the block-quantized (not super-block) types
at column counts that are multiples of 32 only.

Weights are packed GGUF bytes whose codes and scales are distributed as those
of a trained matrix (zero-mean, bell-shaped, scales within a factor of a few of
each other); activations are N(0, 1) with a few large channels.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gollek_amd import tensor_ops as ops

Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = 2, 8, 12, 13, 14
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
TYPE = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}


def listed():
    return [
        # Decode, one sequence.  The smallest call: a key / value projection of
        # grouped-query attention.
        {"name": "matvec_q4_k_1024x4096", "kind": "matvec", "type": "q4_k", "rows": 1024, "cols": 4096, "layers": 1},
        # FFN gate / up projection of eight layers (a token passes every
        # layer's weights once, so they come from HBM).
        {"name": "matvec_q4_k_14336x4096", "kind": "matvec", "type": "q4_k", "rows": 14336, "cols": 4096, "layers": 8},
        # FFN down projection; Q6_K in half the layers of a Q4_K_M file.
        {"name": "matvec_q6_k_4096x14336", "kind": "matvec", "type": "q6_k", "rows": 4096, "cols": 14336, "layers": 8},
        # lm_head of a 128k vocabulary, Q6_K in Q4_K_M files.
        {"name": "matvec_q6_k_128256x4096", "kind": "matvec", "type": "q6_k", "rows": 128256, "cols": 4096, "layers": 1},
        # The Java drop-in's call: float arrays in host memory, synchronous.
        {"name": "host_matvec_q8_0_4096x4096", "kind": "host", "type": "q8_0", "rows": 4096, "cols": 4096, "layers": 1},
        # Decode of 16 sequences together: gate / up projection of four layers.
        {"name": "gemm_q4_k_m16_14336x4096", "kind": "gemm", "type": "q4_k", "m": 16, "rows": 14336, "cols": 4096, "layers": 4},
        # A prompt of 512 tokens: attention projection.
        {"name": "gemm_q8_0_m512_4096x4096", "kind": "gemm", "type": "q8_0", "m": 512, "rows": 4096, "cols": 4096, "layers": 1},
        # A prompt of ragged length: down projection.
        {"name": "gemm_q6_k_m333_4096x14336", "kind": "gemm", "type": "q6_k", "m": 333, "rows": 4096, "cols": 14336, "layers": 1},
        # A long prompt's chunk: gate / up projection, the largest call.
        {"name": "gemm_q4_k_m2048_14336x4096", "kind": "gemm", "type": "q4_k", "m": 2048, "rows": 14336, "cols": 4096, "layers": 1},
        # A hidden size that is no multiple of 256, where files fall back to
        # the 32-element types: a short prompt.
        {"name": "gemm_q8_0_m100_5760x2880", "kind": "gemm", "type": "q8_0", "m": 100, "rows": 5760, "cols": 2880, "layers": 1},
        # Routed MoE block, decode of 16 sequences: router, experts, combine.
        {"name": "moe_q4_k_t16", "kind": "moe", "type": "q4_k", "down": "q4_k", "experts": 128, "top_k": 8,
         "hidden": 2048, "inter": 768, "tokens": 16, "layers": 1},
        # The same block over a prompt of 256 tokens, Q6_K down rows as in
        # half the layers of a Q4_K_M file.
        {"name": "moe_q4_k_q6_k_t256", "kind": "moe", "type": "q4_k", "down": "q6_k", "experts": 128, "top_k": 8,
         "hidden": 2048, "inter": 768, "tokens": 256, "layers": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matvec", "matvec", "host", "gemm", "gemm", "gemm", "moe", "moe"))
    name = rng.choice(("q4_k", "q4_k", "q5_k", "q6_k", "q8_0", "q4_0"))
    if kind == "moe":
        experts = rng.choice((8, 32, 64, 128))
        case = {"kind": kind, "type": name, "down": name, "experts": experts, "top_k": rng.choice((2, 4, 6, 8)),
                "hidden": 256 * rng.randint(4, 12), "inter": 256 * rng.randint(1, 6), "tokens": _log_int(rng, 1, 512),
                "layers": 1}
        if name in ("q4_k", "q5_k") and rng.random() < 0.5:
            case["down"] = "q6_k"
        return case
    cols = 256 * _log_int(rng, 4, 56)
    if name in ("q8_0", "q4_0") and rng.random() < 0.25:
        cols = 32 * _log_int(rng, 28, 180)
    rows = _log_int(rng, 256, 14336)
    if rng.random() < 0.75:
        rows = max(256, rows // 16 * 16)
    case = {"kind": kind, "type": name, "rows": rows, "cols": cols, "layers": 1}
    if kind == "gemm":
        m = _log_int(rng, 2, 2048)
        # no more than the largest listed call
        case["m"] = max(2, min(m, 2048 * 14336 * 4096 // (rows * cols)))
    return case


# ---- packed GGUF matrices ---------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 17)
    return g


def _uniform(g, shape, lo, hi):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=g)


def _codes(g, shape, sigma, mid, lo, hi):
    """Bell-shaped integer codes around `mid`, as uint8 (two's complement)."""
    v = torch.empty(shape, device="cuda", dtype=torch.float16).normal_(0.0, sigma, generator=g)
    return v.add_(mid).round_().clamp_(lo, hi).to(torch.int16).to(torch.uint8)


def _halves(x):
    return x.to(torch.float16).view(torch.uint8)


def _pack_scales(sc, mn):
    """8 + 8 six-bit codes -> the 12 bytes of a Q4_K / Q5_K super-block."""
    lo = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6)], 1)
    return torch.cat([lo, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)


def _packed_blocks(t, nb, g):
    """(nb, block bytes) uint8 on the GPU."""
    if t == Q8_0:
        d = _uniform(g, (nb, 1), 3e-4, 8e-4)
        return torch.cat([_halves(d), _codes(g, (nb, 32), 40.0, 0.0, -127, 127)], 1)
    if t == Q4_0:
        d = _uniform(g, (nb, 1), 4e-3, 1.2e-2)
        q = _codes(g, (nb, 32), 2.7, 8.0, 0, 15)
        return torch.cat([_halves(d), q[:, :16] | (q[:, 16:] << 4)], 1)
    if t in (Q4_K, Q5_K):
        top = 15 if t == Q4_K else 31
        d = _uniform(g, (nb, 1), 1e-4, 2.4e-4) * (15.0 / top)
        sc = torch.randint(20, 64, (nb, 8), device="cuda", generator=g, dtype=torch.uint8)
        off = torch.randint(-3, 4, (nb, 8), device="cuda", generator=g, dtype=torch.int16)
        mn = (sc.to(torch.int16) + off).clamp_(0, 63).to(torch.uint8)
        q = _codes(g, (nb, 4, 2, 32), top / 5.6, top / 2.0, 0, top)
        parts = [_halves(d), _halves(d * (top / 2.0)), _pack_scales(sc, mn)]
        if t == Q5_K:
            qh = torch.zeros((nb, 32), device="cuda", dtype=torch.uint8)
            for c in range(4):
                for h in range(2):
                    qh |= (q[:, c, h] >> 4) << (2 * c + h)
            parts.append(qh)
            q &= 15
        parts.append((q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128))
        return torch.cat(parts, 1)
    # Q6_K: element 128 h + 32 j + l has ql byte 64 h + 32 (j & 1) + l (nibble
    # j >> 1) and qh byte 32 h + l (bits 2 j, 2 j + 1)
    d = _uniform(g, (nb, 1), 1.5e-5, 4e-5)
    sc = torch.randint(40, 128, (nb, 16), device="cuda", generator=g, dtype=torch.int16)
    sign = torch.randint(0, 2, (nb, 16), device="cuda", generator=g, dtype=torch.int16)
    sc = (sc * (1 - 2 * sign)).to(torch.uint8)
    q = _codes(g, (nb, 2, 4, 32), 10.0, 32.0, 0, 63)
    low, high = q & 15, q >> 4
    ql = torch.stack([low[:, :, 0] | (low[:, :, 2] << 4), low[:, :, 1] | (low[:, :, 3] << 4)], 2)
    qh = high[:, :, 0] | (high[:, :, 1] << 2) | (high[:, :, 2] << 4) | (high[:, :, 3] << 6)
    return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc, _halves(d)], 1)


_PIECE = 1 << 26  # elements generated or decoded at a time


def _packed(t, rows, cols, g):
    be, bb = BLOCK[t]
    nb = rows * (cols // be)
    out = torch.empty((nb, bb), device="cuda", dtype=torch.uint8)
    step = _PIECE // be
    for a in range(0, nb, step):
        out[a:a + step] = _packed_blocks(t, min(step, nb - a), g)
    return out


def _decoded_blocks(t, b):
    """(nb, block elements) float64: the GGUF formats' published decoding."""
    nb = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)

    if t == Q8_0:
        return half(0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    if t == Q4_0:
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1)
        return half(0) * (q.to(torch.float64) - 8.0)
    if t in (Q4_K, Q5_K):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(torch.float64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
        qs = b[:, 16 if t == Q4_K else 48:].reshape(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)
        if t == Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (((b[:, None, 16:48] >> bit) & 1) << 4)
        q = q.to(torch.float64)
        return ((half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)).reshape(nb, 256)
    ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
    parts = [(ql[:, :, j & 1] >> (4 * (j >> 1)) & 15) | ((qh >> (2 * j) & 3) << 4) for j in range(4)]
    q = torch.stack(parts, 2).reshape(nb, 16, 16).to(torch.float64) - 32.0
    sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
    return (half(208) * sc).unsqueeze(2).mul(q).reshape(nb, 256)


def _decoded(t, packed, rows, cols):
    """Float64 rows x cols, in pieces of whole rows: yields (first row, rows)."""
    be = BLOCK[t][0]
    per = cols // be
    step = max(1, _PIECE // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        yield r, _decoded_blocks(t, packed[r * per:(r + n) * per]).reshape(n, cols)


def _activations(g, shape):
    """N(0, 1), one channel in 256 ten times as large."""
    x = torch.empty(shape, device="cuda").normal_(0.0, 1.0, generator=g)
    x[..., ::256] *= 10.0
    return x


# ---- cases ------------------------------------------------------------------

def _inputs(case, seed):
    """What is made from the seed: packed weights and activations."""
    g = _gen(seed)
    t = TYPE[case["type"]]
    if case["kind"] == "moe":
        e, h, i, n = case["experts"], case["hidden"], case["inter"], case["tokens"]
        k = min(case["top_k"], e)
        s = {"gate": _packed(t, e * i, h, g), "up": _packed(t, e * i, h, g),
             "down": _packed(TYPE[case["down"]], e * h, i, g), "x": _activations(g, (n, h)),
             "logits": torch.empty((n, e), device="cuda").normal_(0.0, 1.0, generator=g), "k": k}
        return s
    w = [_packed(t, case["rows"], case["cols"], g) for _ in range(case["layers"])]
    if case["kind"] == "gemm":
        return {"w": w, "x": _activations(g, (case["m"], case["cols"])).to(torch.bfloat16)}
    return {"w": w, "x": _activations(g, (case["cols"],))}


def prepare(case, seed):
    ops.init(0)
    s = _inputs(case, seed)
    s["kind"] = case["kind"]
    t = TYPE[case["type"]]
    torch.cuda.synchronize()
    if case["kind"] == "moe":
        e, h, i, n = case["experts"], case["hidden"], case["inter"], case["tokens"]
        s["n"], s["experts"] = n, e
        s["wg"] = ops.DeviceWeight(t, s["gate"].data_ptr(), e * i, h)
        s["wu"] = ops.DeviceWeight(t, s["up"].data_ptr(), e * i, h)
        s["wd"] = ops.DeviceWeight(TYPE[case["down"]], s["down"].data_ptr(), e * h, i)
        s["ids"] = torch.zeros((n, s["k"]), device="cuda", dtype=torch.int32)
        s["weights"] = torch.zeros((n, s["k"]), device="cuda")
        s["out"] = torch.zeros((n, h), device="cuda")
        s["ws"] = torch.zeros(ops.moe_workspace_bytes(n, s["k"], h, i, e), device="cuda", dtype=torch.uint8)
        return s
    rows, cols = case["rows"], case["cols"]
    if case["kind"] == "host":
        s["x"] = s["x"].cpu().numpy()
        s["tensor"] = ops.GgufTensor("w", (cols, rows), t, s.pop("w")[0].cpu().numpy().reshape(-1))
        s["tensor"].prepare()
        s["y"] = np.zeros(rows, np.float32)
        return s
    s["handles"] = [ops.DeviceWeight(t, w.data_ptr(), rows, cols) for w in s["w"]]
    if case["kind"] == "matvec":
        for w in s["handles"]:  # the layout a program builds once at model load
            w.prepare()
        s["y"] = [torch.zeros(rows, device="cuda") for _ in s["handles"]]
    else:
        s["m"] = case["m"]
        s["y"] = [torch.zeros((case["m"], rows), device="cuda") for _ in s["handles"]]
    return s


def run(state):
    if state["kind"] == "host":
        ops.mat_vec(state["tensor"], state["x"], state["y"])
        return state["y"]
    stream = torch.cuda.current_stream().cuda_stream
    if state["kind"] == "moe":
        ops.moe_block_device(state["wg"], state["wu"], state["wd"], state["experts"], state["x"].data_ptr(),
                             state["logits"].data_ptr(), state["n"], state["k"], ops.ROUTER_SIGMOID,
                             state["ids"].data_ptr(), state["weights"].data_ptr(), state["out"].data_ptr(),
                             state["ws"].data_ptr(), state["ws"].numel(), stream)
        return {"out": state["out"], "weights": state["weights"], "ids": state["ids"]}
    x = state["x"].data_ptr()
    for w, y in zip(state["handles"], state["y"]):
        if state["kind"] == "matvec":
            w.matvec(x, y.data_ptr(), stream=stream)
        else:
            w.gemm_bf16(x, state["m"], y.data_ptr(), stream=stream)
    return state["y"]


def work(case):
    if case["kind"] == "moe":
        e, h, i, n = case["experts"], case["hidden"], case["inter"], case["tokens"]
        k = min(case["top_k"], e)
        touched = e * (1.0 - (1.0 - k / e) ** n)  # experts with a route, expected
        be, bb = BLOCK[TYPE[case["type"]]]
        de, db = BLOCK[TYPE[case["down"]]]
        weights = touched * i * h * (2.0 * bb / be + db / de)
        return {"bytes": weights + 4.0 * n * (2 * h + e + 2 * k), "flops": 6.0 * n * k * h * i}
    be, bb = BLOCK[TYPE[case["type"]]]
    rows, cols, m = case["rows"], case["cols"], case.get("m", 1)
    x = m * cols * (2 if case["kind"] == "gemm" else 4)
    return {"bytes": case["layers"] * (rows * cols * bb / be + x + 4.0 * m * rows),
            "flops": 2.0 * case["layers"] * m * rows * cols}


def tolerance(case):
    # 32-bit sums of exactly decoded weights; measured against exact() over
    # the listed and drawn cases, about four times the largest seen.
    if case["kind"] == "moe":
        return {"rel": 2e-5, "max": 2e-4, "differ": 1e-4}
    return {"rel": 1e-5, "max": 2e-4}


def exact(case, seed):
    s = _inputs(case, seed)
    t = TYPE[case["type"]]
    if case["kind"] != "moe":
        x = s["x"].to(torch.float64).reshape(-1, case["cols"])
        ys = []
        for w in s["w"]:
            y = torch.empty((x.shape[0], case["rows"]), device="cuda", dtype=torch.float64)
            for r, d in _decoded(t, w, case["rows"], case["cols"]):
                y[:, r:r + d.shape[0]] = x @ d.t().contiguous()
            ys.append(y if case["kind"] == "gemm" else y[0])
        return ys[0] if case["kind"] == "host" else ys
    e, h, i, n, k = case["experts"], case["hidden"], case["inter"], case["tokens"], s["k"]
    x = s["x"].to(torch.float64)
    p = torch.sigmoid(s["logits"].to(torch.float64))
    top, ids = torch.topk(p, k, dim=1)
    weights = top / top.sum(1, keepdim=True)
    out = torch.zeros((n, h), device="cuda", dtype=torch.float64)
    for ex in range(e):
        tok, rank = (ids == ex).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        m = {}
        for key, ty, rows, cols in (("gate", t, i, h), ("up", t, i, h), ("down", TYPE[case["down"]], h, i)):
            per = rows * (cols // BLOCK[ty][0])
            m[key] = _decoded_blocks(ty, s[key][ex * per:(ex + 1) * per]).reshape(rows, cols).t().contiguous()
        a = x[tok] @ m["gate"]
        y = (a * torch.sigmoid(a) * (x[tok] @ m["up"])) @ m["down"]
        out.index_add_(0, tok, y * weights[tok, rank].unsqueeze(1))
    return {"out": out, "weights": weights, "ids": None}
