"""What a user of this library has it compute, and how each of those calls is made.

One case = one pass through :class:`cudaintro_amd.Handle` (the quantized layers: the row quantizer
and the GEMM, the two-layer network: both layers) with the outputs in buffers the caller keeps, as
a serving loop or the GEMM suite keeps them.  All matrices are row-major and lie packed.
"""
from __future__ import annotations

import math

import torch

import cudaintro_amd as ci

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # the smallest call: a layer head of a small network, no size a multiple of anything; what
        # it takes is the host path, the launches and one pass through a short kernel
        dict(name="bf16_small_odd", op="gemm", dtype="bf16", M=33, N=250, K=333),
        # small square fp32 product
        dict(name="f32_512", op="gemm", dtype="f32", M=512, N=512, K=512),
        # decode of one token through a bf16 layer: the weights are read once
        dict(name="bf16_decode_1", op="gemm", dtype="bf16", M=1, N=8192, K=8192),
        # decode of eight sequences through a quantized layer: activations quantized per row, int8
        # weights with a scale per output channel, bf16 out
        dict(name="i8_decode_8", op="qlinear", M=8, N=8192, K=8192),
        # a batch between decode and prefill: as many bytes as flops
        dict(name="bf16_batch_256", op="gemm", dtype="bf16", M=256, N=8192, K=8192),
        # the GEMM suite's own size, half precision
        dict(name="f16_4096", op="gemm", dtype="f16", M=4096, N=4096, K=4096),
        # the largest product: the size the bf16 rate is quoted at
        dict(name="bf16_8192", op="gemm", dtype="bf16", M=8192, N=8192, K=8192),
        # an odd width (a vocabulary, a class count): no row of B or C is aligned
        dict(name="bf16_odd", op="gemm", dtype="bf16", M=4096, N=4095, K=4096),
        # fp32 with every size odd
        dict(name="f32_odd", op="gemm", dtype="f32", M=4095, N=4097, K=4099),
        # int8 with one scale per matrix, fp32 out, both operands as the suite stores them
        dict(name="i8_4096_dequant", op="i8", layout="kn", out="f32", scales="tensor",
             M=4096, N=4096, K=4096),
        # prefill of a quantized layer: 2048 tokens, activations quantized on the way in
        dict(name="i8_linear_2048", op="qlinear", M=2048, N=11008, K=4096),
        # the digit classifier's forward pass over a third of its training set: two fp32 layers
        dict(name="mnist_forward", op="mlp", M=20000, K=784, H=512, N=10),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A feature count: mostly a multiple of 64, else whatever comes."""
    v = _log_int(rng, lo, hi)
    return max(64, v // 64 * 64) if rng.random() < 0.6 else v


def draw(rng):
    while True:
        op = rng.choice(["f32", "f32", "bf16", "bf16", "f16", "i8", "i8", "qlinear", "mlp"])
        M, N, K = _log_int(rng, 1, 8192), _width(rng, 64, 16384), _width(rng, 64, 16384)
        if op == "mlp":
            case = dict(op="mlp", M=_log_int(rng, 64, 20000), K=_width(rng, 64, 2048),
                        H=_width(rng, 64, 1024), N=rng.randint(2, 64))
        elif op == "qlinear":
            case = dict(op="qlinear", M=M, N=N, K=K)
        elif op == "i8":
            case = dict(op="i8", layout=rng.choice(["kn", "nk"]),
                        out=rng.choice(["i32", "f32", "bf16"]),
                        scales=rng.choice(["tensor", "vector"]), M=M, N=N, K=K)
        else:
            case = dict(op="gemm", dtype=op, M=M, N=N, K=K)
        f32 = op in ("f32", "mlp")
        w = work(case)
        if w["flops"] <= (1.37e11 if f32 else 5.5e11) and w["bytes"] <= 6e8:
            return case


class State:
    pass


def _normal(g, rows, cols, dtype=torch.float32, sigma=1.0):
    x = torch.randn((rows, cols), generator=g, device="cuda", dtype=torch.float32)
    if sigma != 1.0:
        x *= sigma
    return x.to(dtype)


def _uniform(g, rows, cols, lo=-1.0, hi=1.0):
    return torch.rand((rows, cols), generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = State()
    s.h, s.op = ci.Handle(), case["op"]
    M, N, K = case["M"], case["N"], case["K"]
    if s.op == "gemm":
        s.dtype = case["dtype"]
        if s.dtype == "f32":
            s.A, s.B = _uniform(g, M, K), _uniform(g, K, N)
        else:
            # activations N(0, 1); weights N(0, 0.02) where the call is a layer's (fewer rows than
            # columns by far), N(0, 1) for a plain product
            s.A = _normal(g, M, K, TORCH[s.dtype])
            s.B = _normal(g, K, N, TORCH[s.dtype], 0.02 if 16 * M <= N else 1.0)
        s.out = torch.empty((M, N), dtype=TORCH[s.dtype], device="cuda")
    elif s.op == "i8":
        s.layout = ci.B_NK if case["layout"] == "nk" else ci.B_KN
        shape = (N, K) if case["layout"] == "nk" else (K, N)
        s.A = torch.randint(-127, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
        s.B = torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)
        s.kind = case["out"]
        if s.kind == "i32":
            s.out = torch.empty((M, N), dtype=torch.int32, device="cuda")
        else:
            s.out_type = ci.OUT_BF16 if s.kind == "bf16" else ci.OUT_F32
            s.out = torch.empty((M, N), device="cuda",
                                dtype=torch.bfloat16 if s.kind == "bf16" else torch.float32)
            vec = case["scales"] == "vector"
            s.sa = _uniform(g, 1, M if vec else 1, 0.5 / 127, 1.5 / 127).reshape(-1)
            s.sb = _uniform(g, 1, N if vec else 1, 0.5 / 127, 1.5 / 127).reshape(-1)
    elif s.op == "qlinear":
        s.x = _normal(g, M, K)
        s.wq, s.sw = s.h.quantize_rows_i8(_normal(g, N, K, sigma=0.02))
        s.xq = torch.empty((M, K), dtype=torch.int8, device="cuda")
        s.sx = torch.empty((M,), dtype=torch.float32, device="cuda")
        s.out = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    else:
        H = case["H"]
        s.x = _uniform(g, M, K, 0.0, 1.0)  # pixel intensities
        s.w1, s.w2 = _normal(g, K, H, sigma=math.sqrt(2 / K)), _normal(g, H, N, sigma=math.sqrt(2 / H))
        s.b1, s.b2 = _normal(g, 1, H, sigma=0.1).reshape(-1), _normal(g, 1, N, sigma=0.1).reshape(-1)
        s.hidden = torch.empty((M, H), dtype=torch.float32, device="cuda")
        s.out = torch.empty((M, N), dtype=torch.float32, device="cuda")
    return s


def run(s):
    h = s.h
    if s.op == "gemm":
        return {"f32": h.gemm_f32, "f16": h.gemm_f16, "bf16": h.gemm_bf16}[s.dtype](s.A, s.B, out=s.out)
    if s.op == "i8":
        if s.kind == "i32":
            return h.gemm_i8_i32(s.A, s.B, s.layout, out=s.out)
        return h.gemm_i8_dequant(s.A, s.B, s.sa, s.sb, s.layout, s.out_type, out=s.out)
    if s.op == "qlinear":
        h.quantize_rows_i8(s.x, out=(s.xq, s.sx))
        h.gemm_i8_dequant(s.xq, s.wq, s.sx, s.sw, ci.B_NK, ci.OUT_BF16, out=s.out)
        return s.out, s.xq, s.sx
    h.linear_f32(s.x, s.w1, s.b1, ci.ACT_RELU, out=s.hidden)
    h.linear_f32(s.hidden, s.w2, s.b2, ci.ACT_NONE, out=s.out)
    return s.hidden, s.out


def work(case):
    """Every input read once, every output (the activations handed to the next step are outputs
    too) written once and read once by the step after it."""
    M, N, K = case["M"], case["N"], case["K"]
    if case["op"] == "gemm":
        e = SIZE[case["dtype"]]
        return {"bytes": e * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if case["op"] == "i8":
        o = 2 if case["out"] == "bf16" else 4
        return {"bytes": M * K + K * N + o * M * N, "flops": 2 * M * N * K}
    if case["op"] == "qlinear":
        return {"bytes": 4 * M * K + 2 * M * K + N * K + 2 * M * N + 8 * M + 4 * N,
                "flops": 2 * M * N * K}
    H = case["H"]
    return {"bytes": 4 * (M * K + K * H + H + 2 * M * H + H * N + N + M * N),
            "flops": 2 * M * H * (K + N)}


def tolerance(case):
    """int8: the sums, the quantizer and the scaling are defined to the bit.  Floating sums: four
    times what the results differ by from the same products summed in 64 bits (and rounded once:
    the last bit of a 16-bit result may fall the other way)."""
    if case["op"] in ("i8", "qlinear"):
        return "exact"
    dtype = case.get("dtype", "f32")
    if dtype == "bf16":
        return {"rel": 6.6e-3, "max": 1.6e-2}
    if dtype == "f16":
        return {"rel": 8.4e-4, "max": 2e-3}
    return {"rel": 1e-5, "max": 1e-4}  # K = 4099: 1.1e-6 and 1.1e-5, and growing with K
