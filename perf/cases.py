"""Performance cases of the ConvRot int4 / int8 linears.

A case is one call (or the four calls of a block) that a diffusion model's
forward, or the loader in front of it, makes through the package's public
functions: the W4A4 linear with and without a LoRA, the W8A8 linear, and the
weight quantizer with its inverse.  Activations are N(0, 1) with 1% of the
channels scaled by 20, weights N(0, 0.02) in fp16 as the loader quantizes them,
biases fp16 as the layers keep them.
"""
from __future__ import annotations

import importlib
import math

import torch

_PKG = "comfyui-int4-convrot-rdna4_amd"
_int4 = importlib.import_module(_PKG + "._int4")
_int8 = importlib.import_module(_PKG + "._int4.int8_eager")

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_ES = {"bf16": 2, "f16": 2, "f32": 4}

# the four linears of a double-stream block of hidden size 3072: (K, N)
_BLOCK = ((3072, 9216), (3072, 3072), (3072, 12288), (12288, 3072))


def _w4(name, M, K, N, G=256, dtype="bf16", rank=0, bias=True):
    return {"name": name, "kind": "w4a4", "M": M, "K": K, "N": N, "G": G, "dtype": dtype, "rank": rank, "bias": bias}


def listed():
    return [
        # one conditioning vector through a layer (a time or modulation embedding): launches and weight bytes
        _w4("w4a4_vector_m1", 1, 3072, 3072),
        # a short prompt's token stream, the single-linear configuration of the tests
        _w4("w4a4_m256", 256, 3072, 3072),
        # the text stream of a double-stream block with a LoRA attached
        _w4("w4a4_txt_qkv_lora_m512", 512, 3072, 9216, rank=32),
        # the image stream's long rows with a LoRA attached
        _w4("w4a4_img_mlp_down_lora_m4096", 4096, 12288, 3072, rank=32),
        # the headline: the four linears of a block at 4096 image + 512 text tokens
        {"name": "w4a4_block_m4608", "kind": "block", "M": 4608, "G": 256, "dtype": "bf16"},
        # a large image (or a batch) through the widest layer of the token sweep
        _w4("w4a4_large_m16384", 16384, 3840, 15360),
        # an odd resolution in a model that runs in fp16
        _w4("w4a4_ragged_f16_m1333", 1333, 2304, 6912, dtype="f16"),
        # a hidden size that is no multiple of 128: 64-wide rotation groups, the packed int4 kernels
        _w4("w4a4_k1600_m1024", 1024, 1600, 4800, G=64),
        # layers kept at int8 by the precision policy: the image stream and the text stream
        {"name": "w8a8_img_mlp_up_m4096", "kind": "w8a8", "M": 4096, "K": 3072, "N": 12288, "G": 256,
         "dtype": "bf16", "bias": True},
        {"name": "w8a8_txt_mlp_down_m512", "kind": "w8a8", "M": 512, "K": 12288, "N": 3072, "G": 256,
         "dtype": "bf16", "bias": True},
        # a layer quantized on load: fp16 weight -> codes and scales -> the GEMM's operand
        {"name": "quantize_weight_12288x3072", "kind": "quantize", "N": 12288, "K": 3072, "G": 256, "bits": 4},
        # its inverse, as the sensitivity scoring runs it on every layer
        {"name": "dequantize_weight_12288x3072", "kind": "dequantize", "N": 12288, "K": 3072, "G": 256, "bits": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: 1 to 16384 tokens, widths 512 to 12288, heights 512 to 15360, every rotation group."""
    kind = rng.choice(("w4a4", "w4a4", "w4a4", "w4a4", "w8a8", "quantize", "dequantize"))
    G = rng.choice((256, 256, 256, 64, 16))
    bits = 8 if kind == "w8a8" else rng.choice((4, 4, 8)) if kind != "w4a4" else 4
    # widths: mostly multiples of 256, else of the rotation group (int4 codes are packed by groups of 64)
    unit = (G if bits == 8 else max(G, 64)) if rng.random() < 0.4 else 256
    K = max(1, round(_log_int(rng, 512, 12288) / unit)) * unit
    N = _log_int(rng, 512, 15360)
    if rng.random() < 0.7:
        N = max(1, round(N / 64)) * 64
    if kind in ("quantize", "dequantize"):
        while N * K > 12288 * 3072:
            N = max(1, N // 2)
        return {"kind": kind, "N": N, "K": K, "G": G, "bits": bits}
    M = _log_int(rng, 1, 16384)
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
    # no dearer than the largest listed case: int8 products and wider outputs cost twice
    # as much as int4 ones in bf16, the row-major kernels four times
    tiled = _tiled_bytes(N, K, bits) > 0
    share = 4 if not tiled else 2 if kind == "w8a8" or dtype != "bf16" else 1
    while share * M * N * K > 16384 * 3840 * 15360:
        M //= 2
    case = {"kind": kind, "M": M, "K": K, "N": N, "G": G, "dtype": dtype, "bias": rng.random() < 0.8}
    if kind == "w4a4":
        case["rank"] = rng.choice((0, 0, 32, 64)) if case["dtype"] != "f32" else 0
    return case


# --------------------------------------------------------------------------
# inputs (made from the seed alone, on the GPU)
# --------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _activations(M, K, dtype, seed, salt=1):
    g = _gen(seed, salt)
    x = torch.randn((1, M, K), generator=g, device="cuda")
    channels = torch.randperm(K, generator=g, device="cuda")[:max(1, round(0.01 * K))]
    x[..., channels] *= 20.0
    return x.to(_DT[dtype])


def _weight(N, K, seed, salt=2):
    return (torch.randn((N, K), generator=_gen(seed, salt), device="cuda") * 0.02).to(torch.float16)


def _bias(N, seed, salt=3):
    return (torch.randn((N,), generator=_gen(seed, salt), device="cuda") * 0.01).to(torch.float16)


def _lora(N, K, R, seed):
    g = _gen(seed, 4)
    return ((torch.randn((R, K), generator=g, device="cuda") * 0.02).to(torch.bfloat16),
            (torch.randn((N, R), generator=g, device="cuda") * 0.02).to(torch.bfloat16))


def _linear_state(case, seed, salt=0):
    M, K, N, G = case["M"], case["K"], case["N"], case["G"]
    w = _weight(N, K, seed, salt + 2)
    st = {"x": _activations(M, K, case["dtype"], seed, salt + 1), "G": G,
          "bias": _bias(N, seed, salt + 3) if case.get("bias") else None, "lora": None, "tiled": None}
    if case["kind"] == "w8a8":
        st["q"], st["s"] = _int8.quantize_convrot_w8a8_weight(w, G)
        st["tiled"] = _int4.prepare_convrot_w8a8_weight_i8t(st["q"])
    else:
        st["q"], st["s"] = _int4.quantize_convrot_w4a4_weight(w, G)
        st["tiled"] = _int4.prepare_convrot_w4a4_weight_bf6(st["q"])
        if case.get("rank"):
            st["lora"] = _lora(N, K, case["rank"], seed)
    return st


def _block_cases(case):
    return [dict(case, kind="w4a4", K=K, N=N, bias=True, rank=0) for K, N in _BLOCK]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "block":
        return {"kind": kind, "layers": [_linear_state(c, seed, 10 * (i + 1)) for i, c in enumerate(_block_cases(case))]}
    if kind in ("quantize", "dequantize"):
        st = {"kind": kind, "bits": case["bits"], "G": case["G"]}
        w = _weight(case["N"], case["K"], seed)
        if kind == "quantize":
            st["w"] = w
        elif case["bits"] == 4:
            st["q"], st["s"] = _int4.quantize_convrot_w4a4_weight(w, case["G"])
        else:
            st["q"], st["s"] = _int8.quantize_convrot_w8a8_weight(w, case["G"])
        return st
    return dict(_linear_state(case, seed), kind=kind)


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def _w4a4(st):
    return _int4.convrot_w4a4_linear(st["x"], st["q"], st["s"], bias=st["bias"], convrot_groupsize=st["G"],
                                     lora=st["lora"], qweight_bf6=st["tiled"])


def run(state):
    kind = state["kind"]
    if kind == "w4a4":
        return _w4a4(state)
    if kind == "block":
        return [_w4a4(layer) for layer in state["layers"]]
    if kind == "w8a8":
        return _int4.convrot_w8a8_linear(state["x"], state["q"], state["s"], bias=state["bias"],
                                         convrot_groupsize=state["G"], qweight_i8t=state["tiled"])
    G = state["G"]
    if kind == "quantize":
        if state["bits"] == 4:
            q, s = _int4.quantize_convrot_w4a4_weight(state["w"], G)
            tiled = _int4.prepare_convrot_w4a4_weight_bf6(q)
        else:
            q, s = _int8.quantize_convrot_w8a8_weight(state["w"], G)
            tiled = _int4.prepare_convrot_w8a8_weight_i8t(q)
        return [q, s] if tiled is None else [q, s, tiled]
    if state["bits"] == 4:
        return _int4.dequantize_convrot_w4a4_weight(state["q"], state["s"], G)
    return _int8.dequantize_convrot_w8a8_weight(state["q"], state["s"], G)


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

def _tiled_bytes(N, K, bits):
    rows = (N + 255) // 256 * 256
    if bits == 4:
        return rows * K * 3 // 4 if K % 128 == 0 else 0
    return rows * K if K % 64 == 0 else 0


def work(case):
    kind = case["kind"]
    if kind == "block":
        parts = [work(c) for c in _block_cases(case)]
        return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}
    K, N = case["K"], case["N"]
    bits = 8 if kind == "w8a8" else case.get("bits", 4)
    codes = N * K * bits // 8
    # the rotation of n values is n log2(G) additions
    if kind == "quantize":
        return {"bytes": 2 * N * K + codes + 4 * N + _tiled_bytes(N, K, bits), "flops": N * K * math.log2(case["G"])}
    if kind == "dequantize":
        return {"bytes": codes + 4 * N + 4 * N * K, "flops": N * K * math.log2(case["G"])}
    M, R, es = case["M"], case.get("rank", 0), _ES[case["dtype"]]
    weight = _tiled_bytes(N, K, bits) or codes
    return {"bytes": es * M * K + weight + 4 * N + (2 * N if case.get("bias") else 0) + 2 * R * (K + N) + es * M * N,
            "flops": 2 * M * N * K + M * K * math.log2(case["G"]) + 2 * M * R * (K + N)}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"              # codes, their tiling and the scales' 16-bit values
    if kind == "dequantize":
        return {"rel": 2e-6}        # 32-bit sums of one rotation group
    # the codes are whole numbers and their products exact: what is left is the
    # fp32 epilogue and its one rounding to the output type (2-norm 2^-9.3 of bf16,
    # 2^-12.3 of f16), and with a LoRA the 16-bit rounding of its inner product
    if case["dtype"] == "bf16":
        return {"rel": 7e-3}
    if case["dtype"] == "f16":
        return {"rel": 1.5e-3 if case.get("rank") else 1e-3}
    return {"rel": 1e-6}


# --------------------------------------------------------------------------
# the same results in 64 bits, plain torch
# --------------------------------------------------------------------------

def _hadamard(G):
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device="cuda")
    h = h4
    while h.shape[0] < G:
        h = torch.kron(h, h4)
    return h / math.sqrt(G)


def _rotate(x, G):
    rows, K = x.shape
    return (x.double().reshape(-1, G) @ _hadamard(G)).reshape(rows, K)


def _round(v, dtype):
    """float64 values rounded once to a 16- or 32-bit type, kept in float64."""
    bits, low = {"bf16": (8, -133), "f16": (11, -24), "f32": (24, -149)}[dtype]
    _, e = torch.frexp(v)
    e = torch.clamp(e.to(torch.int64) - bits, min=low)
    step = ((e + 1023) << 52).view(torch.float64)     # 2^e to the last bit, which ldexp on a GPU does not promise
    return torch.round(v / step) * step


def _quantize(x, G, dtype, qmax):
    """(codes, scales) in float64: the row scale and the quotient take the input's type."""
    xr = _round(_rotate(x, G), dtype)
    floor = _round(torch.tensor(1e-10, dtype=torch.float64, device="cuda"), dtype)
    a = torch.maximum(xr.abs().amax(dim=1, keepdim=True), floor)
    s = _round((a / qmax).float().double(), dtype)
    z = _round((xr / s).float().double(), dtype)
    return torch.clamp(torch.nan_to_num(torch.round(z)), -qmax, qmax), s


def _exact_linear(case, seed, salt=0):
    K, N, G = case["K"], case["N"], case["G"]
    qmax = 127 if case["kind"] == "w8a8" else 7
    x = _activations(case["M"], K, case["dtype"], seed, salt + 1)[0]
    qx, sx = _quantize(x, G, case["dtype"], qmax)
    qw, sw = _quantize(_weight(N, K, seed, salt + 2), G, "f16", qmax)
    y = (qx @ qw.t()) * sx * sw.reshape(1, -1)
    if case.get("bias"):
        y += _bias(N, seed, salt + 3).double()
    if case.get("rank"):
        down, up = _lora(N, K, case["rank"], seed)
        y += (x.double() @ down.double().t()) @ up.double().t()
    return y.unsqueeze(0)


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        return [_exact_linear(c, seed, 10 * (i + 1)) for i, c in enumerate(_block_cases(case))]
    if kind in ("w4a4", "w8a8"):
        return _exact_linear(case, seed)
    qmax = 7 if case["bits"] == 4 else 127
    q, s = _quantize(_weight(case["N"], case["K"], seed), case["G"], "f16", qmax)
    if kind == "quantize":
        if case["bits"] == 4:
            n = q.to(torch.int32) & 15
            q = (n[:, ::2] | (n[:, 1::2] << 4)).to(torch.uint8).view(torch.int8)
        out = [q.to(torch.int8), s.reshape(-1)]
        return out + [None] if _tiled_bytes(case["N"], case["K"], case["bits"]) else out
    # H is symmetric and its own inverse
    return _rotate(q * s, case["G"])
