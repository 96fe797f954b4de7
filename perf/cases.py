"""The calls this library's time is spent on, as a program that uses it makes them.

Each case is one public entry point of `lighthouse_amd.ops` at one size: GEMMs in 16 bit, f32 and fp8
(large, odd, decode), fused attention, row-wise kernels, the nanoGPT block and the GPT forward.
`listed()` names the twelve that stand for the rest, `draw()` gives others of the same ranges,
`prepare` / `run` / `work` / `tolerance` make, run, price and judge a case.
"""

import math

import torch

from lighthouse_amd import ops

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1}
LARGEST_GEMM = 2 * 4096**3       # flops of the largest 16-bit and f32 products
LARGEST_FP8 = 2 * 8192**3
LARGEST_ATTENTION = 4 * 64 * 2048 * 2048 * 128
LARGEST_ROWWISE = 64 * 1024 * 1024
ROWS_FORWARD = 8192              # B T of the largest forward


def _gemm(name, dtype, M, N, K, *, layout="nn", epilogue="none", out="same"):
    return {"name": name, "kind": "gemm", "dtype": dtype, "M": M, "N": N, "K": K, "layout": layout,
            "epilogue": epilogue, "out": out}


def _attention(name, dtype, Z, H, T, d, causal):
    return {"name": name, "kind": "attention", "dtype": dtype, "Z": Z, "H": H, "T": T, "d": d, "causal": causal}


def _gpt(name, kind, dtype, B, T, C, *, variant="gelu", layers=0, vocab=0):
    return {"name": name, "kind": kind, "dtype": dtype, "B": B, "T": T, "C": C, "variant": variant, "layers": layers,
            "vocab": vocab}


def listed():
    return [
        # The large 16-bit product: a prefill-sized or training-sized matrix multiplication.
        _gemm("gemm_bf16_4096", "bf16", 4096, 4096, 4096),
        # Sizes nobody tuned for: rows that are not 16-byte aligned, a K that is no multiple of a
        # k-step, with the fused bias + ReLU of a payload layer.
        _gemm("gemm_f16_odd", "f16", 1000, 4097, 1000, epilogue="bias_relu"),
        # The f32 payload of the reference's own tests, with its fused epilogue.
        _gemm("gemm_f32_1024", "f32", 1024, 1024, 1024, epilogue="bias_relu"),
        # The quantised product and its decode shape (one token of each of 16 sequences).
        _gemm("gemm_fp8_8192", "fp8", 8192, 8192, 8192, out="bf16"),
        _gemm("gemm_fp8_decode", "fp8", 16, 8192, 8192, out="bf16"),
        # Prefill attention of a decoder.
        _attention("attention_bf16_causal", "bf16", 4, 16, 2048, 64, True),
        # Attention over a short batch of a length that no tile divides.
        _attention("attention_f16_ragged", "f16", 2, 3, 1000, 64, False),
        # A normalisation on its own, bound by memory.
        {"name": "layer_norm_f32", "kind": "rowwise", "op": "layer_norm", "dtype": "f32", "M": 8192, "N": 768},
        # One transformer block at the benchmark's size, and the reference's own small block (f16,
        # separate q / k / v projections, ReLU, not causal), where latency and launches count.
        _gpt("block_bf16", "block", "bf16", 8, 1024, 768),
        _gpt("block_f16_small", "block", "f16", 1, 256, 256, variant="reference"),
        # A whole model: the forward over one prompt of odd length, which each new token costs
        # (there is no key / value cache), and over a full batch of contexts, as an evaluation runs it.
        _gpt("forward_bf16_prompt", "forward", "bf16", 1, 100, 768, layers=12, vocab=50257),
        _gpt("forward_bf16_batch", "forward", "bf16", 8, 1024, 768, layers=12, vocab=50257),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A size spread over the logarithm of lo .. hi: half of them multiples of 64 (where that fits),
    a quarter multiples of 8, a quarter as they come."""
    n, how = _log_uniform(rng, lo, hi), rng.random()
    if how < 0.5 and n >= 64:
        return n // 64 * 64
    if how < 0.75 and n >= 8:
        return n // 8 * 8
    return n


def _draw_gemm(rng, lo_m, lo, hi, largest):
    while True:
        M, N, K = _size(rng, lo_m, hi), _size(rng, lo, hi), _size(rng, lo, hi)
        if 2 * M * N * K <= largest:
            return M, N, K


def draw(rng):
    kind = rng.choice(["gemm16", "gemm16", "gemm32", "fp8", "fp8", "attention", "attention", "rowwise", "block", "block",
                       "forward", "forward"])
    if kind == "gemm16":
        M, N, K = _draw_gemm(rng, 1, 64, 8192, LARGEST_GEMM)
        case = _gemm("", rng.choice(["bf16", "f16"]), M, N, K, layout=rng.choice(["nn", "nn", "nt", "tn"]),
                     epilogue=rng.choice(["none", "bias", "bias_relu", "bias_gelu"]), out=rng.choice(["same", "same", "f32"]))
    elif kind == "gemm32":
        M, N, K = _draw_gemm(rng, 32, 32, 4096, LARGEST_GEMM)
        case = _gemm("", "f32", M, N, K, layout=rng.choice(["nn", "nn", "nt"]), epilogue=rng.choice(["none", "bias_relu"]))
    elif kind == "fp8":
        M, N, K = _draw_gemm(rng, 1, 128, 8192, LARGEST_FP8)
        case = _gemm("", "fp8", M, N, K, out=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "attention":
        while True:
            Z, H, T, d = rng.randint(1, 8), rng.randint(1, 16), _size(rng, 64, 4096), rng.choice([64, 64, 64, 128, 96, 32])
            if 4 * Z * H * T * T * d <= LARGEST_ATTENTION:
                break
        case = _attention("", rng.choice(["bf16", "bf16", "f16", "f32"]), Z, H, T, d, rng.random() < 0.5)
    elif kind == "rowwise":
        while True:
            M, N = _size(rng, 16, 16384), _size(rng, 64, 50257)
            if M * N <= LARGEST_ROWWISE:
                break
        case = {"kind": "rowwise", "op": rng.choice(["layer_norm", "softmax", "gelu"]), "dtype": rng.choice(["f32", "bf16"]),
                "M": M, "N": N}
    elif kind == "block":
        case = _gpt("", "block", rng.choice(["bf16", "f16", "f32"]), rng.randint(1, 8), _size(rng, 16, 1024),
                    rng.choice([256, 512, 768, 1024]), variant=rng.choice(["gelu", "gelu", "reference"]))
    else:
        while True:
            B, T = rng.randint(1, 8), _size(rng, 2, 1024)
            if B * T <= ROWS_FORWARD:
                break
        case = _gpt("", "forward", rng.choice(["bf16", "f16"]), B, T, rng.choice([256, 512, 768]), layers=rng.randint(1, 12),
                    vocab=_size(rng, 256, 50257))
    case.pop("name", None)  # (a drawn case has none)
    return case


def _quantised(x):
    """Per-tensor quantisation: scale = amax / 448, codes = e4m3(x / scale)."""
    scale = float(x.abs().max()) / 448.0
    return (x / scale).to(torch.float8_e4m3fn), scale


def _block_weights(case, randn):
    """Weights N(0, 0.02) in the matmul type, [in, out]; LayerNorm in f32; the reference's variant
    has separate bias-free q / k / v projections and f32 biases."""
    C, dt = case["C"], DTYPES[case["dtype"]]
    reference = case["variant"] == "reference"
    weights = {"w_o": (C, C), "w_fc": (C, 4 * C), "w_proj": (4 * C, C)}
    weights.update({"w_q": (C, C), "w_k": (C, C), "w_v": (C, C)} if reference else {"w_qkv": (C, 3 * C)})
    p = {k: (randn(*s) * 0.02).to(dt) for k, s in weights.items()}
    for k, n in (("b_o", C), ("b_fc", 4 * C), ("b_proj", C)) + (() if reference else (("b_qkv", 3 * C),)):
        p[k] = (randn(n) * 0.02).to(torch.float32 if reference else dt)
    for k in ("ln1", "ln2"):
        p[k + "_g"], p[k + "_b"] = 1.0 + 0.1 * randn(C), 0.02 * randn(C)
    return p


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, device="cuda", generator=g)

    s = dict(case)
    kind = case["kind"]
    if kind == "gemm" and case["dtype"] == "fp8":
        s["a"], s["scale_a"] = _quantised(randn(case["M"], case["K"]))
        s["b"], s["scale_b"] = _quantised(randn(case["K"], case["N"]))
        s["out_dtype"] = DTYPES[case["out"]]
    elif kind == "gemm":
        dt = DTYPES[case["dtype"]]
        out = dt if case["out"] == "same" else DTYPES[case["out"]]
        ta, tb = case["layout"] == "tn", case["layout"] == "nt"
        M, N, K = case["M"], case["N"], case["K"]

        def operand(*shape):  # the f32 payload's operands are uniform in [-1, 1], the 16-bit ones N(0, 1)
            if dt == torch.float32:
                return torch.rand(shape, device="cuda", generator=g) * 2 - 1
            return randn(*shape).to(dt)

        s["a"] = operand(K, M) if ta else operand(M, K)
        s["b"] = operand(N, K) if tb else operand(K, N)
        s["options"] = {"out_dtype": out, "transpose_a": ta, "transpose_b": tb, "relu": case["epilogue"] == "bias_relu",
                        "gelu": case["epilogue"] == "bias_gelu"}
        s["bias"] = None if case["epilogue"] == "none" else operand(N).to(out)
    elif kind == "attention":
        s["q"], s["k"], s["v"] = (randn(case["Z"], case["H"], case["T"], case["d"]).to(DTYPES[case["dtype"]]) for _ in range(3))
    elif kind == "rowwise":
        s["x"] = randn(case["M"], case["N"]).to(DTYPES[case["dtype"]])
        if case["op"] == "layer_norm":
            s["gamma"], s["beta"] = 1.0 + 0.1 * randn(case["N"]), 0.02 * randn(case["N"])
    else:
        B, T, C = case["B"], case["T"], case["C"]
        dt, reference = DTYPES[case["dtype"]], case["variant"] == "reference"
        s["x"] = randn(B, T, C)
        s["heads"] = C // 64
        s["options"] = {"causal": not reference, "activation": "relu" if reference else "gelu_tanh"}
        if kind == "block":
            s["params"] = _block_weights(case, randn)
            need = ops.nanogpt_block_workspace_bytes(B, T, C, dt, bias_dtype=torch.float32 if reference else None, **s["options"])
            s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
        else:
            s["layers"] = [_block_weights(case, randn) for _ in range(case["layers"])]
            s["lnf_g"], s["lnf_b"] = 1.0 + 0.1 * randn(C), 0.02 * randn(C)
            s["lm_w"] = (randn(C, case["vocab"]) * 0.02).to(dt)
    return s


def run(s):
    kind = s["kind"]
    if kind == "gemm" and s["dtype"] == "fp8":
        return ops.gemm_fp8(s["a"], s["b"], s["scale_a"], s["scale_b"], out_dtype=s["out_dtype"])
    if kind == "gemm":
        return ops.gemm(s["a"], s["b"], s["bias"], **s["options"])
    if kind == "attention":
        return ops.attention(s["q"], s["k"], s["v"], causal=s["causal"])
    if kind == "rowwise":
        if s["op"] == "layer_norm":
            return ops.layer_norm(s["x"], s["gamma"], s["beta"])
        return ops.softmax(s["x"]) if s["op"] == "softmax" else ops.gelu_tanh(s["x"])
    if kind == "block":
        return ops.nanogpt_block(s["x"], s["params"], s["heads"], workspace=s["workspace"], **s["options"])
    return ops.nanogpt_forward(s["x"], s["layers"], s["lnf_g"], s["lnf_b"], s["lm_w"], None, s["heads"], **s["options"])


def work(case):
    kind = case["kind"]
    e = BYTES[case["dtype"]]
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        out = e if case["out"] == "same" else BYTES[case["out"]]
        bias = 0 if case["epilogue"] == "none" else N * out
        return {"bytes": (M * K + K * N) * e + M * N * out + bias, "flops": 2 * M * N * K}
    if kind == "attention":
        Z, H, T, d = case["Z"], case["H"], case["T"], case["d"]
        pairs = T * (T + 1) // 2 if case["causal"] else T * T
        return {"bytes": 4 * Z * H * T * d * e, "flops": 4 * Z * H * pairs * d}
    if kind == "rowwise":
        per_element = {"layer_norm": 7, "softmax": 5, "gelu": 7}[case["op"]]
        return {"bytes": 2 * case["M"] * case["N"] * e, "flops": per_element * case["M"] * case["N"]}
    B, T, C = case["B"], case["T"], case["C"]
    pairs = T * T if case["variant"] == "reference" else T * (T + 1) // 2
    layers = 1 if kind == "block" else case["layers"]
    flops = layers * (24 * B * T * C * C + 4 * B * pairs * C)
    size = layers * 12 * C * C * e + B * T * C * 4
    if kind == "block":
        return {"bytes": size + B * T * C * 4, "flops": flops}
    return {"bytes": size + C * case["vocab"] * e + B * T * case["vocab"] * 4, "flops": flops + 2 * B * T * C * case["vocab"]}


# About four times what each kind shows against the same computation in 64 bits (relative 2-norm, and
# largest difference over the larger of the value and the result's root mean square): one rounding of
# the result for the 16-bit products, the roundings of the intermediate values for attention, block and
# forward, the order of the sums for f32 results, and the matrix cores' own fp8 accumulation (1.5e-5).
TOLERANCE = {
    ("gemm", "bf16"): (7e-3, 1.6e-2), ("gemm", "f16"): (8.5e-4, 2e-3), ("gemm", "f32"): (4.4e-6, 3.4e-5),
    ("gemm", "16 bit to f32"): (1.3e-6, 1.2e-5), ("gemm", "fp8 to f32"): (6e-5, 8.7e-4),
    ("attention", "bf16"): (1.2e-2, 2.4e-1), ("attention", "f16"): (1.5e-3, 2.8e-2), ("attention", "f32"): (2.4e-6, 4.1e-5),
    ("rowwise", "bf16"): (7e-3, 1.6e-2), ("rowwise", "f32"): (3.6e-7, 1.6e-6),
    ("block", "bf16"): (5e-3, 2.4e-2), ("block", "f16"): (6e-4, 3e-3), ("block", "f32"): (2.4e-6, 1.9e-5),
    ("forward", "bf16"): (1.3e-2, 6.2e-2), ("forward", "f16"): (1.6e-3, 8e-3),
}


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "gemm" and dtype == "fp8":
        dtype = "bf16" if case["out"] == "bf16" else "fp8 to f32"
    elif kind == "gemm" and dtype != "f32" and case["out"] == "f32":
        dtype = "16 bit to f32"
    rel, largest = TOLERANCE[kind, dtype]
    return {"rel": rel, "max": largest}
