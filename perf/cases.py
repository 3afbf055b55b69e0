"""The work a user of this package has it do, as cases that can be timed and compared.

A case is one projection out = act(x) . W^T through `GemmPlan.run`: x[M, K] are the tokens in
flight, W[N, K] the weights a program keeps.  16-bit operands go straight in; for the byte dtypes
the weights were quantised when they were loaded and the activations, which the previous layer
leaves in bf16, are quantised on the device in every pass in front of the product -- that is
what an fp8 or MXFP4 layer costs its user.

Fields of a case: M, N, K; dtype = "f16" | "bf16" | "fp8_e4m3" | "mxfp4" (operands), out = "f32" |
"bf16" | "f16"; bias; weights = "rows" (row-major, as a checkpoint holds them) or "k8"
(pre-shuffled once when loaded, for MXFP4 with the activations' scale bytes in lane order).
"""
from __future__ import annotations

import math

import torch

from aster_amd import quantize
from aster_amd.gemm import GemmPlan

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_BITS = {"f16": 16, "bf16": 16, "fp8_e4m3": 8, "mxfp4": 4}

# (N, K) of the projections the tests, the benchmark and the shape sweep use: square ones, up- and
# down-projections, with rows that are whole slices (4096, 8192, 14336, 28672) and one whose rows
# are not (11008)
_PROJECTIONS = ((4096, 4096), (14336, 4096), (11008, 4096), (28672, 4096), (4096, 14336),
                (4096, 11008), (8192, 8192), (1024, 8192), (8192, 28672))


def _case(M, N, K, dtype, out, bias=False, weights="rows", name=None):
    c = {"M": M, "N": N, "K": K, "dtype": dtype, "out": out, "bias": bias, "weights": weights}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest product anyone calls the library for (the fp16 known-answer size of the
        # tests): launch and host latency
        _case(256, 256, 256, "f16", "f32", name="f16_256"),
        # a layer whose sizes are no multiple of anything: ragged rows, odd N (a classifier head), bias
        _case(777, 1001, 1032, "bf16", "bf16", bias=True, name="bf16_odd_bias"),
        # one sequence decoding: a whole weight matrix is read for one token
        _case(1, 14336, 4096, "bf16", "bf16", name="bf16_decode_m1"),
        # a full decoding batch on the same weights
        _case(64, 14336, 4096, "bf16", "bf16", name="bf16_decode_m64"),
        # a small batch through a down-projection whose rows are no whole number of slices
        _case(7, 4096, 11008, "bf16", "bf16", name="bf16_decode_down"),
        # decoding on fp8 weights, the activations quantised per tensor in the pass
        _case(16, 14336, 4096, "fp8_e4m3", "bf16", name="fp8_decode_m16"),
        # decoding on MXFP4 weights through a down-projection
        _case(16, 4096, 14336, "mxfp4", "bf16", name="mxfp4_decode_down"),
        # a prompt of as many tokens as its user typed
        _case(333, 14336, 4096, "bf16", "bf16", name="bf16_prompt_333"),
        # a prompt through an fp8 down-projection
        _case(500, 4096, 14336, "fp8_e4m3", "bf16", name="fp8_prompt_down"),
        # the f16 -> f32 shape the reference publishes a figure for
        _case(2048, 4096, 4096, "f16", "f32", name="f16_2048x4096x4096"),
        # a long prefill on MXFP4, weights and scale planes laid out once when loaded
        _case(4096, 14336, 4096, "mxfp4", "bf16", weights="k8", name="mxfp4_prefill"),
        # the benchmark's headline: a large compute-bound product
        _case(8192, 8192, 8192, "bf16", "bf16", name="bf16_8192"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: small products, decoding, prompts, long prefills, a quarter each."""
    kind = rng.choice(("small", "decode", "prompt", "large"))
    if kind == "small":
        dtype = rng.choice(("f16", "bf16"))
        return _case(_log_int(rng, 16, 1200), _log_int(rng, 16, 1200), 8 * _log_int(rng, 4, 256),
                     dtype, rng.choice(("f32", dtype)), bias=rng.random() < 0.5)
    dtype = rng.choice(("bf16", "bf16", "f16", "fp8_e4m3", "mxfp4"))
    N, K = rng.choice(_PROJECTIONS)
    out = "f16" if dtype == "f16" else "bf16"
    bias = rng.random() < 0.25
    if kind == "decode":
        return _case(_log_int(rng, 1, 64), N, K, dtype, out, bias)
    M = _log_int(rng, 65, 2047) if kind == "prompt" else _log_int(rng, 2048, 8192)
    M = min(M, 8192 ** 3 // (N * K))         # no more work than the largest listed case
    weights = "rows"
    if rng.random() < 0.3 and not (dtype == "mxfp4" and K % 512):
        weights = "k8"                       # a program that lays weights out pads its rows too
        M = max(16, M // 16 * 16)
    return _case(M, N, K, dtype, out, bias, weights)


def prepare(case, seed):
    """Weights (quantised and laid out), activations, output and plan: all of it from the seed."""
    M, N, K, dtype, k8 = case["M"], case["N"], case["K"], case["dtype"], case["weights"] == "k8"
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    src = torch.float16 if dtype == "f16" else torch.bfloat16
    x = torch.randn(M, K, generator=g, device=dev, dtype=torch.float32).to(src)
    w = (torch.randn(N, K, generator=g, device=dev, dtype=torch.float32) * 0.02).to(src)
    s = {"case": dict(case), "x": x,
         "out": torch.zeros(M, N, device=dev, dtype=_TORCH[case["out"]]),
         "bias": torch.randn(N, generator=g, device=dev) if case["bias"] else None}
    u8 = dict(device=dev, dtype=torch.uint8)
    if dtype == "fp8_e4m3":
        s["w"], s["w_scale"] = torch.zeros(N, K, **u8), torch.zeros(1, device=dev)
        s["xq"], s["x_scale"] = torch.zeros(M, K, **u8), torch.zeros(1, device=dev)
        quantize.quantize_fp8_tensor_device(w.data_ptr(), N * K, s["w"].data_ptr(),
                                            s["w_scale"].data_ptr(), src_dtype="bf16")
    elif dtype == "mxfp4":
        s["w"], s["w_scale"] = torch.zeros(N, K // 2, **u8), torch.zeros(N, K // 32, **u8)
        # lane order pads the scale bytes to groups of 128 rows
        s["xq"] = torch.zeros(M, K // 2, **u8)
        s["x_scale"] = torch.zeros((M + 127) // 128 * 128 if k8 else M, K // 32, **u8)
        quantize.quantize_mxfp4_device(w.data_ptr(), N, K, s["w"].data_ptr(),
                                       s["w_scale"].data_ptr(), src_dtype="bf16")
    else:
        s["w"] = w
    if k8:
        rows, mx = s["w"], s["w_scale"] if dtype == "mxfp4" else None
        s["w"] = torch.zeros_like(rows)
        if mx is not None:
            s["w_scale"] = torch.zeros_like(mx)
        quantize.preshuffle_device(rows.data_ptr(), s["w"].data_ptr(), N, K, dtype, "direct_b_k8",
                                   d_mx_src=mx.data_ptr() if mx is not None else None,
                                   d_mx_dst=s["w_scale"].data_ptr() if mx is not None else None)
        torch.cuda.synchronize()             # `rows` and `mx` are freed on return
    s["plan"] = GemmPlan.create(M, N, K, dtype, case["out"], has_bias=case["bias"],
                                operand_path="direct_b_k8" if k8 else "lds",
                                mx_a_layout="lanes128" if k8 and dtype == "mxfp4" else "rows")
    torch.cuda.synchronize()
    return s


def run(state):
    s, c = state, state["case"]
    bias = s["bias"].data_ptr() if c["bias"] else None
    if c["dtype"] == "fp8_e4m3":
        quantize.quantize_fp8_tensor_device(s["x"].data_ptr(), c["M"] * c["K"], s["xq"].data_ptr(),
                                            s["x_scale"].data_ptr(), src_dtype="bf16")
        s["plan"].run(s["xq"].data_ptr(), s["w"].data_ptr(), s["out"].data_ptr(),
                      scale_a=s["x_scale"].data_ptr(), scale_b=s["w_scale"].data_ptr(), bias=bias)
        return s["out"], s["xq"], s["x_scale"]
    if c["dtype"] == "mxfp4":
        layout = "lanes128" if c["weights"] == "k8" else "rows"
        quantize.quantize_mxfp4_device(s["x"].data_ptr(), c["M"], c["K"], s["xq"].data_ptr(),
                                       s["x_scale"].data_ptr(), src_dtype="bf16",
                                       scales_layout=layout)
        s["plan"].run(s["xq"].data_ptr(), s["w"].data_ptr(), s["out"].data_ptr(),
                      mx_a=s["x_scale"].data_ptr(), mx_b=s["w_scale"].data_ptr(), bias=bias)
        return s["out"], s["xq"], s["x_scale"]
    s["plan"].run(s["x"].data_ptr(), s["w"].data_ptr(), s["out"].data_ptr(), bias=bias)
    return s["out"]


def work(case):
    """Activations (16-bit, as they arrive), weights with their scales, bias: read once; the
    output and, for the byte dtypes, the quantised activations: written once."""
    M, N, K, bits = case["M"], case["N"], case["K"], _BITS[case["dtype"]]
    n = 2 * M * K + N * K * bits // 8 + M * N * (4 if case["out"] == "f32" else 2)
    if bits < 16:
        n += M * K * bits // 8 + ((M + N) * (K // 32) if bits == 4 else 8)
    return {"bytes": n + (4 * N if case["bias"] else 0), "flops": 2 * M * N * K}


def tolerance(case):
    """Against the same operands multiplied in float64 the outputs are off by their own rounding
    (rel 1.7e-3 and at most 3.9e-3 in bf16, 2.1e-4 and 4.9e-4 in f16) or, in f32, by the fp32 sums
    (rel 4.1e-7, at most 2.9e-6 at K = 4096): four times that.  The quantised activations are
    bytes and stay the same."""
    if case["out"] == "f32":
        return {"rel": 1.6e-6, "max": 1.2e-5}
    if case["out"] == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 6.7e-3, "max": 1.6e-2}
