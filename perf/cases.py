"""What the framework is timed on: the calls a quantized-inference program
makes, from one small GEMV to a full prefill GEMM, through the public entry
points (the operators of kernel_craft_torch_ops, and the C ABI's chain call
with its arguments laid out once, as a native decode loop holds them).

Shapes are those of the repository's benchmark and tests (Llama-3-8B layers:
hidden 4096, QKV 6144, gate/up 28672, FFN 14336; the 70B layer 8192 x 28672)
and generic ragged ones.  Weights and activations have the distributions the
tests use: uniform nibbles, zero points and group scales; normal activations
with a few large channels.
"""
from __future__ import annotations

import ctypes
import os
import sys

import torch

# The working folder is the root of the tree that is measured.
sys.path.insert(0, os.path.join(os.getcwd(), "kernel-craft_amd", "python"))

import kernel_craft_torch_ops as kc_ops  # noqa: E402

DEV = "cuda:0"
EPS = 1e-5
F8 = torch.float8_e4m3fn


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one token through the attention output projection: the smallest
        # call of a decode step, launch and host latency weigh as much as
        # the 9 MB of weights
        dict(name="gemv_o_proj", kind="gemv", x="bf16", rows=4096, cols=4096, gs=128),
        # the reference's blocking fp32 operator on a ragged layer with small
        # groups (5120 is no multiple of 2048, 11001 rows)
        dict(name="gemv_f32_ragged", kind="gemv", x="f32", rows=11001, cols=5120, gs=64),
        # RMSNorm and the gate/up projection of one token in one call
        dict(name="norm_gemv_gate_up", kind="gemv", x="norm", rows=28672, cols=4096, gs=128),
        # the four projections of a decode layer from one native call
        dict(name="decode_layer", kind="chain", hidden=4096, kv=1024, ffn=14336, gs=128),
        # batched decode: 16 sequences through the down projection, weights
        # as the checkpoint converter writes them
        dict(name="gemm_int4_down_m16", kind="gemm", m=16, rows=4096, cols=14336, gs=128,
             shuffled=False),
        # the largest decode batch on the large layer, weights laid out for
        # the matrix cores once at load time
        dict(name="gemm_int4_m64", kind="gemm", m=64, rows=28672, cols=8192, gs=128, shuffled=True),
        # weights to fp32 for an ordinary matmul (prefill with the
        # reference's operators)
        dict(name="int4_dequantize", kind="dequant", rows=14336, cols=4096, gs=128),
        # fp32 activations to FP8 and back through the reference's blocking
        # operators (its example's round trip)
        dict(name="fp8_round_trip", kind="round_trip", rows=4096, cols=4096),
        # calibrating and quantizing one layer: statistics of X and W,
        # then both quantizers; a ragged token count
        dict(name="smoothquant_layer", kind="smooth", tokens=2003, rows=14336, cols=4096),
        # a W8A8 linear layer on a decode batch: RMSNorm + quantization of
        # the tokens, then the FP8 GEMM
        dict(name="w8a8_qkv_decode", kind="w8a8", tokens=32, rows=6144, cols=4096),
        # a chunk of a prompt through the FP8 down projection
        dict(name="fp8_gemm_chunk", kind="fp8_gemm", m=1000, rows=4096, cols=14336, out="bf16"),
        # a full prefill batch on the large layer
        dict(name="fp8_gemm_prefill", kind="fp8_gemm", m=16384, rows=28672, cols=8192, out="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _rows(rng, lo, hi):
    """Output features: mostly multiples of 128, sometimes any number."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.3 else max(lo, n // 128 * 128)


def _cols(rng, lo, hi, step):
    """Input features: multiples of 1024 half of the time, else of `step`."""
    k = _log_int(rng, lo, hi)
    return max(lo, k // 1024 * 1024 if rng.random() < 0.5 else k // step * step)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "chain", "gemm", "gemm", "dequant", "round_trip", "smooth",
                       "w8a8", "w8a8", "fp8_gemm", "fp8_gemm"])
    if kind == "gemv":
        x = rng.choice(["bf16", "f32", "norm"])
        return dict(kind=kind, x=x, rows=_rows(rng, 1024, 28672), cols=_cols(rng, 1024, 16384, 128),
                    gs=rng.choice([128, 128, 64, 32]))
    if kind == "chain":
        hidden = 512 * rng.randint(4, 16)
        return dict(kind=kind, hidden=hidden, kv=hidden // rng.choice([1, 4, 8]),
                    ffn=256 * int(hidden * rng.uniform(2.6, 3.6) / 256), gs=rng.choice([128, 128, 64]))
    if kind == "gemm":
        shuffled = rng.random() < 0.5
        return dict(kind=kind, m=_log_int(rng, 2, 64), rows=_rows(rng, 1024, 28672),
                    cols=_cols(rng, 1024, 14336, 128),
                    gs=128 if shuffled else rng.choice([128, 128, 64]), shuffled=shuffled)
    if kind == "dequant":
        return dict(kind=kind, rows=_rows(rng, 512, 28672), cols=_cols(rng, 1024, 8192, 128),
                    gs=rng.choice([128, 64, 32]))
    if kind == "round_trip":
        return dict(kind=kind, rows=_log_int(rng, 16, 8192), cols=_cols(rng, 1024, 14336, 8))
    if kind == "smooth":
        return dict(kind=kind, tokens=_log_int(rng, 128, 16384), rows=_rows(rng, 1024, 28672),
                    cols=_cols(rng, 1024, 8192, 8))
    if kind == "w8a8":
        return dict(kind=kind, tokens=_log_int(rng, 1, 64), rows=_rows(rng, 1024, 28672),
                    cols=_cols(rng, 1024, 8192, 16))
    return dict(kind=kind, m=_log_int(rng, 65, 8192), rows=_rows(rng, 1024, 28672),
                cols=_cols(rng, 1024, 14336, 16), out=rng.choice(["bf16", "bf16", "f32"]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (2 ** 62) + 1)


def _int4(g, rows, cols, gs):
    """Packed nibbles, group scales, zero-point bytes (rows * ceil(G/2) bytes,
    which the kernels index at a row stride of floor(G/2))."""
    G = cols // gs
    packed = torch.randint(0, 256, (rows, cols // 2), dtype=torch.uint8, device=DEV, generator=g)
    scales = torch.rand(rows, G, device=DEV, generator=g) * 0.015 + 0.005
    zeros = torch.randint(0, 256, (rows, (G + 1) // 2), dtype=torch.uint8, device=DEV, generator=g)
    return packed, scales, zeros


def _activations(g, rows, cols, dtype=torch.bfloat16):
    """N(0, 1) with about one channel in 128 fifty times larger."""
    x = torch.randn(rows, cols, device=DEV, generator=g)
    x *= torch.where(torch.rand(cols, device=DEV, generator=g) < 1 / 128, 50.0, 1.0)
    return x.to(dtype)


def _codes(x):
    """Per-row E4M3 codes (int8) and scales of a float matrix."""
    s = x.abs().amax(1) / 448.0
    return (x / s[:, None]).to(F8).view(torch.int8), s


def _weight_codes(g, rows, cols):
    q = torch.empty(rows, cols, dtype=torch.int8, device=DEV)
    s = torch.empty(rows, device=DEV)
    for r in range(0, rows, 4096):
        w = torch.randn(min(4096, rows - r), cols, device=DEV, generator=g) * 0.02
        q[r:r + 4096], s[r:r + 4096] = _codes(w)
    return q, s


def _layer(case):
    """The four projections of a decode layer: (rows, cols)."""
    h, kv, ffn = case["hidden"], case["kv"], case["ffn"]
    return [(h + 2 * kv, h), (h, h), (2 * ffn, h), (h, ffn)]


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind == "gemv":
        st["w"] = _int4(g, case["rows"], case["cols"], case["gs"])
        st["x"] = _activations(g, 1, case["cols"],
                               torch.float32 if case["x"] == "f32" else torch.bfloat16)[0]
        if case["x"] == "norm":
            st["gamma"] = (torch.rand(case["cols"], device=DEV, generator=g) + 0.5).bfloat16()
    elif kind == "chain":
        shapes = _layer(case)
        st["ops"] = []
        for rows, cols in shapes:
            w = _int4(g, rows, cols, case["gs"])
            x = torch.randn(cols, device=DEV, generator=g).bfloat16()
            st["ops"].append((*w, x, torch.empty(rows, dtype=torch.bfloat16, device=DEV)))
        st["table"] = (kc_ops.GemvOp * len(shapes))(*[
            kc_ops.GemvOp(*[t.data_ptr() for t in op], rows, cols, case["gs"], 0)
            for op, (rows, cols) in zip(st["ops"], shapes)])
        st["args"] = (ctypes.cast(st["table"], ctypes.c_void_p), len(shapes),
                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        st["call"] = kc_ops._get_lib().kc_gemv_int4_bf16_chain
    elif kind == "gemm":
        packed, scales, zeros = _int4(g, case["rows"], case["cols"], case["gs"])
        if case["shuffled"]:
            packed = kc_ops.int4_shuffle_mfma(packed, case["rows"], case["cols"])
        st["w"] = (packed, scales, zeros)
        st["x"] = torch.randn(case["m"], case["cols"], device=DEV, generator=g).bfloat16()
    elif kind == "dequant":
        st["w"] = _int4(g, case["rows"], case["cols"], case["gs"])
    elif kind == "round_trip":
        st["x"] = _activations(g, case["rows"], case["cols"], torch.float32)
    elif kind == "smooth":
        st["x"] = _activations(g, case["tokens"], case["cols"])
        st["wt"] = (torch.randn(case["rows"], case["cols"], device=DEV, generator=g) * 0.02).bfloat16()
    elif kind == "w8a8":
        st["h"] = _activations(g, case["tokens"], case["cols"])
        st["gamma"] = (torch.rand(case["cols"], device=DEV, generator=g) + 0.5).bfloat16()
        st["qw"], st["sw"] = _weight_codes(g, case["rows"], case["cols"])
    else:
        st["qx"], st["sx"] = _codes(_activations(g, case["m"], case["cols"], torch.float32))
        st["qw"], st["sw"] = _weight_codes(g, case["rows"], case["cols"])
        st["out"] = torch.bfloat16 if case["out"] == "bf16" else torch.float32
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "gemv":
        if c["x"] == "norm":
            return kc_ops.rmsnorm_int4_gemv_bf16(st["x"], st["gamma"], *st["w"], c["rows"], c["cols"],
                                                 c["gs"], EPS)
        fn = kc_ops.int4_gemv if c["x"] == "f32" else kc_ops.int4_gemv_bf16
        return fn(*st["w"], st["x"], c["rows"], c["cols"], c["gs"])
    if kind == "chain":
        if st["call"](*st["args"]):
            raise RuntimeError(kc_ops.last_error())
        return [op[4] for op in st["ops"]]
    if kind == "gemm":
        fn = kc_ops.int4_gemm_bf16_shuffled if c["shuffled"] else kc_ops.int4_gemm_bf16
        return fn(*st["w"], st["x"], c["rows"], c["cols"], c["gs"])
    if kind == "dequant":
        return kc_ops.int4_dequantize(*st["w"], c["rows"], c["cols"], c["gs"])
    if kind == "round_trip":
        q, s = kc_ops.fp8_quantize(st["x"], per_token=True)
        return q, s, kc_ops.fp8_dequantize(q, s, c["rows"], c["cols"], per_token=True)
    if kind == "smooth":
        ax, aw, sm = kc_ops.smoothquant_stats(st["x"], st["wt"])
        return (ax, aw, sm, *kc_ops.fp8_quantize_smooth(st["x"], sm, "div"),
                *kc_ops.fp8_quantize_smooth(st["wt"], sm, "mul"))
    if kind == "w8a8":
        q, s = kc_ops.rmsnorm_fp8_quantize(st["h"], st["gamma"], EPS)
        return q, s, kc_ops.fp8_gemm_w8a8(q, s, st["qw"], st["sw"])
    return kc_ops.fp8_gemm_w8a8(st["qx"], st["sx"], st["qw"], st["sw"], st["out"])


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def _int4_bytes(rows, cols, gs):
    G = cols // gs
    return rows * (cols // 2 + 4 * G + G // 2)


def work(case):
    kind = case["kind"]
    if kind == "chain":
        return dict(bytes=sum(_int4_bytes(r, k, case["gs"]) + 2 * (r + k) for r, k in _layer(case)),
                    flops=sum(2 * r * k for r, k in _layer(case)))
    n, k = case["rows"], case["cols"]
    if kind == "gemv":
        e = 4 if case["x"] == "f32" else 2
        return dict(bytes=_int4_bytes(n, k, case["gs"]) + e * (n + k * (2 if case["x"] == "norm" else 1)),
                    flops=2 * n * k)
    if kind == "gemm":
        return dict(bytes=_int4_bytes(n, k, case["gs"]) + 2 * case["m"] * (n + k),
                    flops=2 * case["m"] * n * k)
    if kind == "dequant":
        return dict(bytes=_int4_bytes(n, k, case["gs"]) + 4 * n * k, flops=2 * n * k)
    if kind == "round_trip":  # fp32 in, codes out; codes in, fp32 out
        return dict(bytes=n * (10 * k + 8), flops=4 * n * k)
    if kind == "smooth":  # X and W read for the statistics, read again and written as codes
        t = case["tokens"]
        return dict(bytes=(t + n) * (5 * k + 4) + 20 * k, flops=6 * (t + n) * k)
    if kind == "w8a8":
        t = case["tokens"]
        return dict(bytes=t * (4 * k + 8) + 2 * k + n * (k + 4) + 2 * t * n, flops=2 * t * n * k)
    m, e = case["m"], 2 if case["out"] == "bf16" else 4
    return dict(bytes=(m + n) * (k + 4) + e * m * n, flops=2 * m * n * k)


def tolerance(case):
    kind = case["kind"]
    if kind in ("dequant", "round_trip", "smooth"):
        return "exact"
    if (kind, case.get("x")) == ("gemv", "f32"):
        return dict(rel=2e-6)   # fp32 sums: 2e-7 to 4e-7 from 64 bits
    if (kind, case.get("out")) == ("fp8_gemm", "f32"):
        return dict(rel=2e-4)   # the matrix core's FP8 sums: about 5e-5 from 64 bits
    return dict(rel=7e-3)       # bf16 results: 1.7e-3 from 64 bits


def _dequant64(w, rows, cols, gs, r0, r1):
    """Rows r0..r1 of the weights in 64 bits."""
    packed, scales, zeros = w
    G = cols // gs
    p = packed[r0:r1].to(torch.int16)
    q = torch.stack((p & 15, p >> 4), 2).reshape(r1 - r0, G, gs)
    g = torch.arange(G, device=DEV)
    zb = zeros.reshape(-1)[(torch.arange(r0, r1, device=DEV) * (G // 2))[:, None] + (g // 2)[None]]
    z = torch.where((g % 2).bool()[None], zb >> 4, zb & 15).double()
    return (((q ^ 8) - 8).double() - z[..., None]).mul_(scales[r0:r1].double()[..., None]).reshape(r1 - r0, cols)


def _matmul_int4(x, w, rows, cols, gs):
    x = x.double().reshape(-1, cols)
    y = torch.cat([x @ _dequant64(w, rows, cols, gs, r, min(r + 4096, rows)).T
                   for r in range(0, rows, 4096)], 1)
    return y


def _matmul_codes(qx, sx, qw, sw):
    x = qx.view(F8).double()
    y = torch.empty(len(qx), len(qw), dtype=torch.float64, device=DEV)
    for r in range(0, len(qw), 4096):
        y[:, r:r + 4096] = x @ qw[r:r + 4096].view(F8).double().T
    return y.mul_(sx.double()[:, None]).mul_(sw.double())


def _quantized64(x):
    """Per-row scales in 64 bits and the E4M3 codes they give."""
    s = x.abs().amax(1) / 448.0
    s = torch.where(s > 0, s, 1.0)
    return (x / s[:, None]).float().to(F8).view(torch.int8), s


def exact(case, seed):
    kind = case["kind"]
    plain = dict(case, shuffled=False) if kind == "gemm" else case
    st = prepare(plain, seed)
    if kind == "chain":
        return [_matmul_int4(op[3], op[:3], r, k, case["gs"])[0]
                for op, (r, k) in zip(st["ops"], _layer(case))]
    n, k = case["rows"], case["cols"]
    if kind == "gemv":
        x, scale = st["x"].double(), 1.0
        if case["x"] == "norm":  # the products are rounded to bf16, the norm is not
            scale = 1.0 / torch.sqrt((x * x).mean() + EPS)
            x = (x * st["gamma"].double()).bfloat16().double()
        return _matmul_int4(x, st["w"], n, k, case["gs"])[0] * scale
    if kind == "gemm":
        return _matmul_int4(st["x"], st["w"], n, k, case["gs"])
    if kind == "dequant":
        return torch.cat([_dequant64(st["w"], n, k, case["gs"], r, min(r + 4096, n))
                          for r in range(0, n, 4096)])
    if kind == "round_trip":
        q, s = _quantized64(st["x"].double())
        return None, s, q.view(F8).double() * s[:, None]
    if kind == "smooth":
        ax, aw = st["x"].double().abs().amax(0), st["wt"].double().abs().amax(0)
        sm = (ax.sqrt() / aw.clamp(min=1e-5).sqrt()).clamp(min=1e-5)
        return (ax, aw, sm, None, (st["x"].double() / sm).abs().amax(1) / 448.0,
                None, (st["wt"].double() * sm).abs().amax(1) / 448.0)
    if kind == "w8a8":
        h = st["h"].double()
        y = (st["gamma"].double() * h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS)).bfloat16()
        q, s = _quantized64(y.double())
        return None, s, _matmul_codes(q, s, st["qw"], st["sw"])
    return _matmul_codes(st["qx"], st["sx"], st["qw"], st["sw"])
