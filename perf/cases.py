"""Performance cases of the NVFP4 path: quantizers, linears and attention through `ac4k_kernel_amd.ops`.

Sizes are those of this repository's benchmark and tests (LLM linears of N = 14336, K = 4096 and its transpose, decode on
N = 28672, K = 8192, the 75600-token tensors with 40 heads of 128, N = 16384 attention) and ragged relatives of them.
`draw` gives further cases of the same ranges."""
import math

import torch

from ac4k_kernel_amd import ops

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _quantize(rows, cols, precision, **kw):
    """One 2-D tensor [rows, cols] quantized along its contiguous dim: an activation in front of a linear."""
    return dict({"kind": "quantize", "lead": 1, "rows": rows, "heads": 1, "cols": cols, "along": "cols", "precision": precision,
                 "swizzle": False}, **kw)


def _linear(m, n, k, **kw):
    """y = x W^T (+ bias), weights quantized beforehand.  activation: "quantized" (in hand already, as when several
    projections share it), "bf16" (quantized in the pass, two calls) or "fused" (quantized in the pass, one call)."""
    return dict({"kind": "linear", "m": m, "n": n, "k": k, "activation": "quantized", "image": False, "bias": "none", "out": "bf16"}, **kw)


def _attention(batch, nq, nkv, heads, dim, **kw):
    return dict({"kind": "attention", "batch": batch, "nq": nq, "nkv": nkv, "heads": heads, "dim": dim, "layout": "BNHD",
                 "precision": "int8+fp8e4m3"}, **kw)


def listed():
    return [
        # activation of a prefill of 8192 tokens in front of an NVFP4 linear
        dict(_quantize(8192, 4096, "nvfp4"), name="quantize_nvfp4_8192x4096"),
        # ragged: a token count and a width that are multiples of nothing the kernels tile by; per-token int8
        dict(_quantize(4001, 5003, "int8"), name="quantize_int8_4001x5003"),
        # V of a 75600-token attention, per-channel scales along the strided token dim (the largest quantize)
        dict(_quantize(75600, 128, "fp8e4m3", heads=40, along="rows", swizzle=True), name="quantize_fp8_v_75600x40x128"),
        # one decoded token: activation quantized in the call, weights streamed from memory
        dict(_linear(1, 28672, 8192, activation="fused"), name="decode_m1_n28672_k8192"),
        # a small decode batch on a narrow weight with a long K
        dict(_linear(16, 4096, 14336), name="linear_m16_n4096_k14336"),
        # a large decode batch / short prompt, static weights kept as a weight image
        dict(_linear(128, 14336, 4096, image=True), name="linear_m128_n14336_k4096_image"),
        # one layer of a prefill: quantize, then linear with bias
        dict(_linear(2048, 14336, 4096, activation="bf16", bias="bf16"), name="prefill_m2048_n14336_k4096"),
        # ragged: no dim is a multiple of a tile; fp32 result with fp32 bias
        dict(_linear(1001, 5003, 2880, bias="fp32", out="fp32"), name="linear_m1001_n5003_k2880_fp32"),
        # a projection over a 75600-token sequence (the largest linear)
        dict(_linear(75600, 5120, 5120, bias="bf16"), name="linear_m75600_n5120_k5120"),
        # long self-attention, default precision, quantizers included (the largest attention)
        dict(_attention(1, 16384, 16384, 40, 128), name="attention_int8_16384x40x128"),
        # self-attention of medium length on NVFP4 operands
        dict(_attention(1, 4096, 4096, 40, 128, precision="nvfp4", layout="BHND"), name="attention_nvfp4_4096x40x128"),
        # short cross-attention with ragged lengths and a small head dim: launches and host time count
        dict(_attention(2, 777, 257, 12, 64), name="attention_int8_cross_777x257x12x64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature dim: mostly a multiple of 128, sometimes of 64 or 8, sometimes odd."""
    w = _log_int(rng, lo, hi)
    step = rng.choice([128, 128, 128, 128, 64, 8, 1])
    return max(lo, w // step * step)


def draw(rng):
    kind = rng.choice(["quantize", "linear", "linear", "attention"])
    if kind == "quantize":
        precision = rng.choice(["nvfp4", "nvfp4", "fp8e4m3", "int8"])
        if rng.random() < 0.4:  # an attention operand [lead, rows, heads, cols]
            cols, heads = rng.choice([40, 64, 96, 100, 128, 128]), rng.choice([1, 3, 8, 12, 40])
            rows = _log_int(rng, 64, 75600)
            return _quantize(rows, cols, precision, heads=heads, lead=rng.choice([1, 1, 2]) if rows < 30000 else 1,
                             along=rng.choice(["rows", "cols"]), swizzle=precision != "int8" and rng.random() < 0.5)
        cols = _width(rng, 256, 14336)
        return _quantize(_log_int(rng, 1, min(75600, 380_000_000 // cols)), cols, precision)
    if kind == "linear":
        n, k = _width(rng, 256, 28672), _width(rng, 256, 14336)
        m = _log_int(rng, 1, min(75600, 1_900_000_000_000 // (n * k)))
        fused = m <= 32 and k % 64 == 0
        activation = rng.choice(["quantized", "bf16", "fused"] if fused else ["quantized", "bf16"])
        return _linear(m, n, k, activation=activation, image=activation != "fused" and k % 128 == 0 and rng.random() < 0.25,
                       bias=rng.choice(["none", "none", "bf16", "fp32"]), out=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    batch, heads, dim = rng.choice([1, 1, 2]), rng.choice([1, 4, 8, 12, 24, 40]), rng.choice([40, 64, 96, 100, 128, 128, 128])
    nq = _log_int(rng, 32, 16384)
    nkv = nq if rng.random() < 0.6 else _log_int(rng, 32, 16384)
    if batch * heads * nq * nkv > 40 * 16384 * 16384:
        batch = 1
    return _attention(batch, nq, nkv, heads, dim, layout=rng.choice(["BNHD", "BHND"]), precision=rng.choice(["int8+fp8e4m3", "nvfp4"]))


def _normal(shape, gen, std=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=gen)


def _activation(shape, gen):
    """N(0, 1) with 0.1 % outliers of twenty times the size, as transformer activations have."""
    x = _normal(shape, gen)
    mask = torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(generator=gen) < 1e-3
    return torch.where(mask, x * 20.0, x).to(torch.bfloat16)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if case["kind"] == "quantize":
        if case["heads"] == 1 and case["lead"] == 1 and case["along"] == "cols":
            state["x"] = _activation((case["rows"], case["cols"]), gen)
            state["dims"] = (0, 1)
        else:
            state["x"] = _activation((case["lead"], case["rows"], case["heads"], case["cols"]), gen)
            state["dims"] = (1, 3) if case["along"] == "cols" else (3, 1)
    elif case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        w = ops.quantize(_normal((n, k), gen, 0.02).to(torch.bfloat16), 0, 1)
        state["w"] = (ops.prepack_weight(w[0], w[1]), w[2]) if case["image"] else w
        x = _activation((m, k), gen)
        state["x"] = ops.quantize(x, 0, 1) if case["activation"] == "quantized" else x
        state["bias"] = None if case["bias"] == "none" else _normal((n,), gen, 0.5).to(_DTYPES[case["bias"]])
    else:
        b, h, d = case["batch"], case["heads"], case["dim"]

        def operand(length):
            shape = (b, length, h, d) if case["layout"] == "BNHD" else (b, h, length, d)
            return _normal(shape, gen)

        # keys share an offset per channel, which is what the default precision takes out before it quantizes them
        offset = _normal((b, 1, h, d) if case["layout"] == "BNHD" else (b, h, 1, d), gen)
        state["q"] = operand(case["nq"]).to(torch.bfloat16)
        state["k"] = (operand(case["nkv"]) + offset).to(torch.bfloat16)
        state["v"] = operand(case["nkv"]).to(torch.bfloat16)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "quantize":
        return ops.quantize(state["x"], *state["dims"], precision=case["precision"], swizzle=case["swizzle"])
    if case["kind"] == "attention":
        return ops.attention(state["q"], state["k"], state["v"], layout=case["layout"], precision=case["precision"])
    x, w, bias = state["x"], state["w"], state["bias"]
    m, n = case["m"], case["n"]
    out = None if case["out"] == "bf16" else torch.empty((m, n), dtype=_DTYPES[case["out"]], device="cuda")
    if case["activation"] == "fused":
        return ops.fused_linear(x, *w, bias, out=out)
    if case["activation"] == "bf16":
        x = ops.quantize(x, 0, 1)
    if case["image"]:
        return ops.linear_prepacked(*x, *w, bias, out=out, n=n)
    return ops.linear(*x, *w, bias, out=out)


def _up(a, b):
    return (a + b - 1) // b * b


def _nvfp4_bytes(rows, k):
    return rows * _up(k, 64) // 2 + _up(k, 64) // 16 * _up(rows, 16)


def work(case):
    if case["kind"] == "quantize":
        planes = case["lead"] * case["heads"]
        n = planes * case["rows"] * case["cols"]
        r, k = (case["rows"], case["cols"]) if case["along"] == "cols" else (case["cols"], case["rows"])
        out = _nvfp4_bytes(r, k) if case["precision"] == "nvfp4" else r * _up(k, 16) + 4 * _up(r, 16)
        return {"bytes": 2 * n + planes * out, "flops": 0}
    if case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        size = {"none": 0, "bf16": 2, "fp16": 2, "fp32": 4}
        x = _nvfp4_bytes(m, k) if case["activation"] == "quantized" else 2 * m * k
        return {"bytes": x + _nvfp4_bytes(n, k) + size[case["bias"]] * n + size[case["out"]] * m * n, "flops": 2 * m * n * k}
    rows = case["batch"] * case["heads"] * (2 * case["nq"] + 2 * case["nkv"])
    return {"bytes": 2 * rows * case["dim"], "flops": 4 * case["batch"] * case["heads"] * case["nq"] * case["nkv"] * case["dim"]}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "linear":
        # rounding of the result type: a 64-bit evaluation differs from it by 1.7e-3, 2.1e-4 and 5e-8
        return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 1e-6}[case["out"]]}
    # the oracle (other order of sums, another exp2) differs by up to 3e-4, single values by up to 0.019: a probability
    # next to a rounding boundary of its quantization goes the other way
    return {"rel": 1.5e-3, "max": 0.08}
