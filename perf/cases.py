"""The library's performance cases: what a program that runs a diffuser's
B1_0 linears on one MI355X has it do, through the Python entry points.

A case is a dict of plain values; `kind` names the call:

  linear     bonsai_b1.linear, fp32 activations -> fp32 outputs (any token
             count; `mode` "auto" or "exact")
  projections  bonsai_b1.linear_batch over small-batch linears that share one
             input: the modulation projections of a diffusion step
  stream     bonsai_b1.linear_batch with epilogues: q/k/v, the gated output
             projection, FF-in with SwiGLU and gated FF-out of one stream of a
             double-stream block, from fp32 activations
  mlp        LayerNorm + modulation -> packed fp16, FF-in writing SwiGLU or
             GELU as FF-out's packed input, gated FF-out
  single     a single-stream block: LayerNorm + modulation -> packed fp16,
             linear1 (fp32 q/k/v columns, MLP columns into linear2's packed
             input), the attention output packed beside them, gated linear2
  quantize   fp32 weights -> packed B1_0 (the encoder)

Activations are N(0, 1); packed weights have Bernoulli(0.5) sign bits and fp16
scales from U[0.005, 0.05], as in bonsai_b1.synth.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent
for _p in (_ROOT, _ROOT / "bonsai.cpp_amd"):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

import bonsai_b1 as b1  # noqa: E402
from bonsai_b1 import synth  # noqa: E402

EPS = 1e-6
# a drawn case costs no more than the largest listed one (`single_block`)
MOST_FLOPS = 1.0e12
MOST_EXACT_FLOPS = 3.0e10


def listed():
    return [
        # one modulation projection of a step: one token, bound by launch and weight latency
        {"name": "one_token", "kind": "linear", "m": 1, "k": 3072, "n": 18432, "mode": "auto", "count": False},
        # the four modulation projections of a step over one conditioning vector
        {"name": "modulations", "kind": "projections", "m": 1, "k": 3072, "n": "18432,18432,9216,6144"},
        # a batch of conditioning vectors through one projection, outputs checked for non-finite values
        {"name": "few_tokens", "kind": "linear", "m": 12, "k": 3072, "n": 9216, "mode": "auto", "count": True},
        # a short prompt's tokens through an attention projection (an odd count)
        {"name": "prompt", "kind": "linear", "m": 77, "k": 3072, "n": 3072, "mode": "auto", "count": False},
        # the parity configuration: 256 tokens through an attention projection
        {"name": "tokens_256", "kind": "linear", "m": 256, "k": 3072, "n": 3072, "mode": "auto", "count": False},
        # the text stream of a double-stream block, one call, checked for non-finite values
        {"name": "text_stream", "kind": "stream", "m": 512, "k": 3072, "h": 9216},
        # the feed-forward of a double-stream block for a 512 x 512 pixel image
        {"name": "mlp_1024", "kind": "mlp", "m": 1024, "k": 3072, "h": 9216, "act": "swiglu"},
        # another model's width and a ragged token count, no multiple of the tuned ones
        {"name": "other_width", "kind": "linear", "m": 1000, "k": 2048, "n": 5504, "mode": "auto", "count": False},
        # the headline GEMM: image tokens through the MLP up-projection, from fp32 activations
        {"name": "image_up", "kind": "linear", "m": 4096, "k": 3072, "n": 12288, "mode": "auto", "count": False},
        # a single-stream block at 64 x 64 latents and 512 text tokens
        {"name": "single_block", "kind": "single", "m": 4608, "k": 3072, "h": 12288, "act": "gelu_tanh"},
        # the bit-exact mode, run to compare with the reference's scalar path
        {"name": "exact_256", "kind": "linear", "m": 256, "k": 3072, "n": 3072, "mode": "exact", "count": False},
        # a checkpoint's MLP weight through the encoder
        {"name": "encode", "kind": "quantize", "k": 3072, "n": 12288, "order": "numpy"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges: token counts 1 to 4608, odd ones
    included; inner widths mostly multiples of 384 (what the diffuser family's
    hidden sizes are), else of 64 (32 in the exact mode and the encoder);
    output widths of any multiple of 8, odd ones now and then."""
    while True:
        kind = rng.choice(["linear", "linear", "linear", "linear", "projections", "stream", "mlp", "single", "exact",
                           "quantize"])
        if kind in ("linear", "exact"):
            exact_mode = kind == "exact"
            m = _log(rng, 1, 16) if rng.random() < 0.3 else _log(rng, 17, 4608)
            if exact_mode:
                m, k = _log(rng, 1, 1024), 32 * _log(rng, 4, 160)
            else:
                k = 384 * _log(rng, 2, 40) if rng.random() < 0.7 else 64 * _log(rng, 6, 128)
            n = 8 * _log(rng, 32, 3456)
            if rng.random() < 0.15:
                n += 2 * rng.randint(0, 3) + 1
            c = {"kind": "linear", "m": m, "k": k, "n": n, "mode": "exact" if exact_mode else "auto",
                 "count": rng.random() < 0.4}
            if work(c)["flops"] <= (MOST_EXACT_FLOPS if exact_mode else MOST_FLOPS):
                return c
        elif kind == "projections":
            k = 256 * _log(rng, 4, 12)
            return {"kind": "projections", "m": _log(rng, 1, 16), "k": k,
                    "n": ",".join(str(k * rng.randint(1, 6)) for _ in range(rng.randint(2, 6)))}
        elif kind == "stream":
            k = 384 * _log(rng, 3, 8)
            c = {"kind": "stream", "m": _log(rng, 20, 2048), "k": k, "h": k * rng.randint(2, 4)}
            if work(c)["flops"] <= MOST_FLOPS:
                return c
        elif kind in ("mlp", "single"):
            k = 384 * _log(rng, 3, 8)
            c = {"kind": kind, "m": _log(rng, 20 if kind == "mlp" else 64, 4608), "k": k, "h": k * rng.randint(2, 4),
                 "act": rng.choice(["swiglu", "gelu_tanh"])}
            if work(c)["flops"] <= MOST_FLOPS:
                return c
        else:
            return {"kind": "quantize", "k": 32 * _log(rng, 8, 480), "n": _log(rng, 64, 12288),
                    "order": rng.choice(["numpy", "sequential"])}


def _widths(case):
    return [int(v) for v in case["n"].split(",")]


def _linears(case):
    """(tokens, inner width, output width) of the case's linears."""
    m, k = case.get("m", 0), case["k"]
    if case["kind"] == "linear":
        return [(m, k, case["n"])]
    if case["kind"] == "projections":
        return [(m, k, n) for n in _widths(case)]
    h = case["h"]
    if case["kind"] == "stream":
        return [(m, k, k)] * 4 + [(m, k, 2 * h), (m, h, k)]
    up = (2 if case["act"] == "swiglu" else 1) * h
    if case["kind"] == "mlp":
        return [(m, k, up), (m, h, k)]
    return [(m, k, 3 * k + up), (m, k + h, k)]


def work(case):
    k = case["k"]
    if case["kind"] == "quantize":
        return {"bytes": case["n"] * k * 4 + case["n"] * k // 32 * 6, "flops": 2 * case["n"] * k}
    lin = _linears(case)
    m = case["m"]
    weights = sum(kk // 32 * 6 * n for _, kk, n in lin)
    flops = sum(2.0 * mm * kk * n for mm, kk, n in lin)
    if case["kind"] in ("linear", "projections"):
        values = m * k + sum(mm * n for mm, _, n in lin)
    elif case["kind"] == "stream":
        # x, attention output and FF input in; the residuals in; q/k/v and both sums out
        values = m * k * (3 + 2 + 3 + 2) + 2 * k
    elif case["kind"] == "mlp":
        values = 3 * m * k + 3 * k         # x and the residual in, the sum out, scale, shift, gate
    else:
        values = m * k * (3 + 3 + 1) + 3 * k   # x, attention output, residual in; q/k/v and the sum out
    return {"bytes": 4 * values + weights, "flops": flops}


def tolerance(case):
    if case["kind"] == "quantize" or case.get("mode") == "exact":
        return "exact"       # bytes, and the reference's scalar order bit for bit
    if case["kind"] in ("linear", "projections"):
        return {"rel": 8e-4}     # activations rounded to fp16 once (2.1e-4 against 64 bits)
    return {"rel": 1.4e-3}       # two such roundings in a row (3.6e-4)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _inputs(case, seed):
    """Every tensor a case reads, from the seed alone."""
    g = _gen(1000003 * seed + 17)

    def act(m, k):
        return torch.randn((m, k), generator=g, device="cuda", dtype=torch.float32)

    def weights(i):
        mm, k, n = _linears(case)[i]
        return synth.device_packed_weights(n, k, 7919 * seed + 31 * i + 5)

    k, m = case["k"], case.get("m", 0)
    if case["kind"] == "quantize":
        return {"w": 0.02 * act(case["n"], k)}
    t = {"w": [weights(i) for i in range(len(_linears(case)))], "x": act(m, k)}
    if case["kind"] in ("stream", "single"):
        t["attn"] = act(m, k)
    if case["kind"] == "stream":
        t["x2"], t["res2"], t["gate2"] = act(m, k), act(m, k), act(1, k)[0]
    if case["kind"] in ("mlp", "single"):
        t["scale"], t["shift"] = 0.3 * act(1, k)[0], 0.3 * act(1, k)[0]
    if case["kind"] in ("stream", "mlp", "single"):
        t["res"], t["gate"] = act(m, k), act(1, k)[0]
    return t


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    k, m, kind = case["k"], case.get("m", 0), case["kind"]

    def empty(rows, cols):
        return torch.empty((rows, cols), device="cuda", dtype=torch.float32)

    if kind == "linear":
        s["out"] = empty(m, case["n"])
        s["bad"] = torch.zeros(1, dtype=torch.int32, device="cuda") if case["count"] else None
    elif kind == "projections":
        s["outs"] = [empty(m, n) for n in _widths(case)]
        s["ops"] = [(s["x"], b1.device_weights(w, k, o.shape[1]), o) for w, o in zip(s["w"], s["outs"])]
    elif kind == "stream":
        h = case["h"]
        # q, k and v as one resident buffer of adjacent row ranges, their outputs adjacent column ranges
        qkv = torch.cat([w.reshape(-1) for w in s["w"][:3]])
        step = k * (k // 32 * 6)
        s["qkv_w"], s["qkv"] = qkv, empty(m, 3 * k)
        s["h1"], s["ff"], s["h2"] = empty(m, k), empty(m, h), empty(m, k)
        s["bad"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        dw = b1.device_weights
        s["ops"] = [(s["x"], dw(qkv[i * step:(i + 1) * step], k, k), s["qkv"][:, i * k:(i + 1) * k]) for i in range(3)]
        s["ops"] += [(s["attn"], dw(s["w"][3], k, k), s["h1"], ("gate_residual", s["gate"], s["res"])),
                     (s["x2"], dw(s["w"][4], k, 2 * h), s["ff"], "swiglu"),
                     (s["ff"], dw(s["w"][5], h, k), s["h2"], ("gate_residual", s["gate2"], s["res2"]))]
    elif kind == "mlp":
        s["p1"] = torch.empty(m * k * 2, dtype=torch.uint8, device="cuda")
        s["p2"] = torch.empty(m * case["h"] * 2, dtype=torch.uint8, device="cuda")
        s["out"] = empty(m, k)
    elif kind == "single":
        s["p1"] = torch.empty(m * k * 2, dtype=torch.uint8, device="cuda")
        s["p2"] = torch.empty(m * (k + case["h"]) * 2, dtype=torch.uint8, device="cuda")
        s["qkv"], s["out"] = empty(m, 3 * k), empty(m, k)
    else:
        s["packed"] = torch.empty((case["n"], k // 32 * 6), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case = s["case"]
    k, m, kind = case["k"], case.get("m", 0), case["kind"]
    if kind == "linear":
        b1.linear(s["x"], s["w"][0], case["n"], out=s["out"], mode=case["mode"], nonfinite=s["bad"])
        return {"out": s["out"], "bad": s["bad"]} if case["count"] else s["out"]
    if kind == "projections":
        b1.linear_batch(s["ops"])
        return s["outs"]
    if kind == "stream":
        b1.linear_batch(s["ops"], nonfinite=s["bad"])
        return {"qkv": s["qkv"], "h1": s["h1"], "h2": s["h2"], "bad": s["bad"]}
    if kind == "quantize":
        return b1.quantize_f32(s["w"], order=case["order"], out=s["packed"])
    h = case["h"]
    up = (2 if case["act"] == "swiglu" else 1) * h
    if kind == "mlp":
        b1.norm_mod(s["x"], s["scale"], s["shift"], EPS, packed=s["p1"])
        b1.linear_packed_f16_to_packed(s["p1"], s["w"][0], k, up, m, 0, case["act"], packed_out=s["p2"])
        return b1.linear_packed_f16_epi(s["p2"], s["w"][1], h, k, m, "gate_residual", gate=s["gate"],
                                        residual=s["res"], out=s["out"])
    # linear2's input is [attention output | MLP], both written straight into its packed rows
    b1.norm_mod(s["x"], s["scale"], s["shift"], EPS, packed=s["p1"])
    b1.linear_packed_f16_to_packed(s["p1"], s["w"][0], k, 3 * k + up, m, 3 * k, case["act"], out=s["qkv"],
                                   packed_out=s["p2"][2 * k:], ldp=k + h)
    b1.pack_act_f16(s["attn"], packed=s["p2"], ldp=k + h)
    b1.linear_packed_f16_epi(s["p2"], s["w"][1], k + h, k, m, "gate_residual", gate=s["gate"], residual=s["res"],
                             out=s["out"])
    return {"qkv": s["qkv"], "out": s["out"]}


# ------------------------------------------------------- 64-bit reference --

def _unpack(raw, n, k):
    """float64 [n, k] of packed B1_0 bytes."""
    blocks = raw.reshape(n, k // 32, 6)
    scale = blocks[:, :, :2].contiguous().view(torch.float16).to(torch.float64)
    bits = torch.arange(8, device=raw.device, dtype=torch.uint8)
    sign = (blocks[:, :, 2:].unsqueeze(-1) >> bits) & 1
    return ((2.0 * sign.to(torch.float64) - 1.0).reshape(n, k // 32, 32) * scale).reshape(n, k)


def _mm(x, raw, n):
    """float64 x @ W^T, over ranges of the weight rows."""
    k = x.shape[1]
    rows = raw.reshape(n, -1)
    step = max(64, (1 << 26) // k)
    return torch.cat([x @ _unpack(rows[i:i + step].contiguous(), min(step, n - i), k).t().contiguous()
                      for i in range(0, n, step)], dim=1)


def _norm(t):
    x = t["x"].double()
    mean = x.mean(dim=1, keepdim=True)
    var = (x - mean).square().mean(dim=1, keepdim=True)
    return (x - mean) / torch.sqrt(var + EPS) * (t["scale"].double() + 1.0) + t["shift"].double()


def _activate(y, act):
    if act == "swiglu":
        half = y.shape[1] // 2
        return torch.nn.functional.silu(y[:, :half]) * y[:, half:]
    return torch.nn.functional.gelu(y, approximate="tanh")


def exact(case, seed):
    t = _inputs(case, seed)
    k, kind = case["k"], case["kind"]
    if kind == "quantize":
        return None      # bytes
    x = t["x"].double()
    if kind == "linear":
        y = _mm(x, t["w"][0], case["n"])
        return {"out": y, "bad": None} if case["count"] else y
    if kind == "projections":
        return [_mm(x, w, n) for w, n in zip(t["w"], _widths(case))]
    h = case["h"]
    if kind == "stream":
        qkv = torch.cat([_mm(x, w, k) for w in t["w"][:3]], dim=1)
        h1 = t["res"].double() + t["gate"].double() * _mm(t["attn"].double(), t["w"][3], k)
        ff = _activate(_mm(t["x2"].double(), t["w"][4], 2 * h), "swiglu")
        h2 = t["res2"].double() + t["gate2"].double() * _mm(ff, t["w"][5], k)
        return {"qkv": qkv, "h1": h1, "h2": h2, "bad": None}
    up = (2 if case["act"] == "swiglu" else 1) * h
    a = _norm(t)
    if kind == "mlp":
        mid = _activate(_mm(a, t["w"][0], up), case["act"])
        return t["res"].double() + t["gate"].double() * _mm(mid, t["w"][1], k)
    y = _mm(a, t["w"][0], 3 * k + up)
    mid = torch.cat([t["attn"].double(), _activate(y[:, 3 * k:], case["act"])], dim=1)
    out = t["res"].double() + t["gate"].double() * _mm(mid, t["w"][1], k)
    return {"qkv": y[:, :3 * k], "out": out}
