"""The work that users of this framework have it do, as cases that can be timed and checked.

Each case is one pass through the public entry points: quantizing activations,
the packed GEMM, the linear layer, dequantizing, and preparing a weight at load
time. Widths and projections are those of this repository's tests and
benchmark, or any multiple of 64; token counts run from one decoded token to a
prefill of 8192.
"""
import torch

import quant_ops_amd as qo
from quant_ops_amd.workloads import orthogonal

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# hidden and FFN widths of the repository's tests, each split by get_decompose_dim
WIDTHS = (1024, 1536, 2048, 2560, 3072, 3584, 4096, 5120, 5632, 6144, 6912, 7168, 8192, 8960, 9216, 9728, 10240, 11008,
          12288, 13696, 13824, 14336, 16384, 18432, 18944, 20480, 22016, 24576, 25600, 27648, 28672)

# (out, in) features of projections over those widths: attention, gate / up, down
PROJECTIONS = ((4096, 4096), (6144, 4096), (14336, 4096), (4096, 14336), (11008, 4096), (4096, 11008), (5120, 5120),
               (13824, 5120), (5120, 13824), (3584, 3584), (18944, 3584), (3584, 18944), (8192, 8192), (28672, 8192),
               (8192, 28672), (1024, 4096), (2048, 2048))

# The largest listed work, which bounds the drawn cases: activations of the
# widest quantize (elements) and the products of the prefill GEMM (M N K).
MOST_ELEMENTS = 8192 * 14336
MOST_PRODUCTS = 4096 * 14336 * 4096


def listed():
    return [
        # float32 activations to int8 codes: the accuracy script's and examples' default type
        {"name": "quant_fp32_128x4096", "kind": "quant", "tokens": 128, "features": 4096, "dtype": "fp32", "clip": 1.0,
         "pack": False},
        # prefill activations of a hidden size of 4096
        {"name": "quant_fp16_2048x4096", "kind": "quant", "tokens": 2048, "features": 4096, "dtype": "fp16", "clip": 0.9,
         "pack": True},
        # the input of the down projection, a large prefill
        {"name": "quant_bf16_8192x14336", "kind": "quant", "tokens": 8192, "features": 14336, "dtype": "bf16",
         "clip": 1.0, "pack": True},
        # a ragged batch at an FFN width whose rows are no multiple of 16 bytes
        {"name": "quant_bf16_1021x18944", "kind": "quant", "tokens": 1021, "features": 18944, "dtype": "bf16",
         "clip": 0.9, "pack": True},
        # a square decomposition (96 x 96), an odd number of tokens, codes as int8
        {"name": "quant_fp16_777x9216", "kind": "quant", "tokens": 777, "features": 9216, "dtype": "fp16", "clip": 1.0,
         "pack": False},
        # gate / up projection of a prefill, weight in the reference's [K/8, N] layout
        {"name": "gemm_4096x14336x4096", "kind": "gemm", "m": 4096, "n": 14336, "k": 4096, "layout": "kn",
         "out": "fp16"},
        # a mixed decode / prefill batch against a smaller FFN's gate projection
        {"name": "gemm_333x11008x4096", "kind": "gemm", "m": 333, "n": 11008, "k": 4096, "layout": "nk", "out": "bf16"},
        # decode of a batch of 16: the down projection
        {"name": "linear_16x4096x14336", "kind": "linear", "m": 16, "n": 4096, "k": 14336, "dtype": "bf16", "clip": 0.9,
         "bias": False},
        # one chunk of a chunked prefill, with bias
        {"name": "linear_512x4096x14336", "kind": "linear", "m": 512, "n": 4096, "k": 14336, "dtype": "bf16",
         "clip": 0.9, "bias": True},
        # a whole prefill through the down projection
        {"name": "linear_4096x4096x14336", "kind": "linear", "m": 4096, "n": 4096, "k": 14336, "dtype": "bf16",
         "clip": 0.9, "bias": False},
        # the decode direction of the codec: packed codes back to float32
        {"name": "dequant_2048x4096", "kind": "dequant", "tokens": 2048, "features": 4096, "packed": True,
         "dtype": "fp16"},
        # loading a weight: pack its codes, convert the layout, unpack again for export
        {"name": "weight_14336x4096", "kind": "weight", "n": 14336, "k": 4096},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _width(rng, most):
    """A width of the tests, or any multiple of 64 (odd decompositions among them)."""
    if rng.random() < 0.7:
        return rng.choice([w for w in WIDTHS if w <= most])
    return 64 * _log(rng, 8, min(most, 16384) // 64)


def draw(rng):
    kind = rng.choices(("quant", "gemm", "linear", "dequant", "weight"), (8, 5, 5, 1, 1))[0]
    if kind == "quant":
        dtype = rng.choices(("bf16", "fp16", "fp32"), (4, 3, 2))[0]
        features = _width(rng, 16384 if dtype == "fp32" else 28672)
        most = (2048 * 16384 if dtype == "fp32" else MOST_ELEMENTS) // features
        return {"kind": kind, "tokens": _log(rng, 1, min(8192, most)), "features": features, "dtype": dtype,
                "clip": rng.choice((1.0, 0.95, 0.9, 0.8)), "pack": rng.random() < 0.8}
    if kind in ("gemm", "linear"):
        n, k = rng.choice(PROJECTIONS)
        if rng.random() < 0.25:   # ragged: any out width, any packed in width
            n, k = _log(rng, 200, 16384), 64 * _log(rng, 8, 224)
        m = _log(rng, 1, min(8192, MOST_PRODUCTS // (n * k)))
        if kind == "gemm":
            return {"kind": kind, "m": m, "n": n, "k": k, "layout": rng.choice(("kn", "nk")),
                    "out": rng.choices(("fp16", "bf16", "fp32"), (5, 4, 1))[0]}
        return {"kind": kind, "m": m, "n": n, "k": k, "dtype": rng.choice(("bf16", "fp16")),
                "clip": rng.choice((1.0, 0.95, 0.9)), "bias": rng.random() < 0.4}
    if kind == "dequant":
        features = _width(rng, 28672)
        return {"kind": kind, "tokens": _log(rng, 1, min(8192, MOST_ELEMENTS // features)), "features": features,
                "packed": rng.random() < 0.7, "dtype": rng.choice(("fp32", "fp16"))}
    n, k = rng.choice(PROJECTIONS)
    if rng.random() < 0.3:
        n, k = _log(rng, 200, 16384), 8 * _log(rng, 64, 1792)
    return {"kind": "weight", "n": n, "k": k}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _words(g, rows, words):
    return torch.randint(-2 ** 31, 2 ** 31, (rows, words), generator=g, dtype=torch.int32, device="cuda")


def _scales(g, n, lo, hi, dtype):
    return (lo + (hi - lo) * torch.rand(n, generator=g, device="cuda")).to(dtype)


def _activations(g, tokens, features, dtype):
    """N(0, 1) with 0.5 % of the channels as outliers, x30."""
    x = torch.randn(tokens, features, generator=g, device="cuda")
    channels = torch.randperm(features, generator=g, device="cuda")[: -(-features // 200)]
    x[:, channels] *= 30.0
    return x.to(dtype)


def _transforms(seed, features, dtype):
    m, n = qo.get_decompose_dim(features)
    return orthogonal(m, 2 * seed + 1, dtype).cuda(), orthogonal(n, 2 * seed + 2, dtype).cuda()


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind == "quant":
        dtype = DTYPES[case["dtype"]]
        s["x"] = _activations(g, case["tokens"], case["features"], dtype)
        s["left"], s["right"] = _transforms(seed, case["features"], dtype)
    elif kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s["a"] = _words(g, m, k // 8)
        s["b"] = _words(g, k // 8, n) if case["layout"] == "kn" else _words(g, n, k // 8).t()
        s["sa"], s["sb"] = _scales(g, m, 0.01, 0.1, torch.float16), _scales(g, n, 0.001, 0.01, torch.float16)
    elif kind == "linear":
        m, n, k, dtype = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
        s["x"] = _activations(g, m, k, dtype)
        s["left"], s["right"] = _transforms(seed, k, dtype)
        s["w"], s["sw"] = _words(g, n, k // 8), _scales(g, n, 0.001, 0.01, torch.float16)
        s["bias"] = torch.randn(n, generator=g, device="cuda").to(dtype) if case["bias"] else None
    elif kind == "dequant":
        t, f = case["tokens"], case["features"]
        s["codes"] = _words(g, t, f // 8) if case["packed"] else torch.randint(
            -8, 8, (t, f), generator=g, dtype=torch.int8, device="cuda")
        s["scales"] = _scales(g, t, 0.01, 3.0, DTYPES[case["dtype"]])
    else:
        s["codes"] = torch.randint(-8, 8, (case["n"], case["k"]), generator=g, dtype=torch.int8, device="cuda")
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "quant":
        return qo.flatquant_dynamic_quantize(s["x"], s["left"], s["right"], case["clip"], case["pack"])
    if kind == "gemm":
        return qo.int4_matmul(s["a"], s["b"], s["sa"], s["sb"], out_dtype=DTYPES[case["out"]])
    if kind == "linear":
        return qo.w4a4_flatquant_linear(s["x"], s["left"], s["right"], s["w"], s["sw"], case["clip"], s["bias"])
    if kind == "dequant":
        return qo.dequantize_int4(s["codes"], s["scales"], case["packed"])
    packed = qo.prepare_w4a4_weight(s["codes"])
    return packed, qo.transpose_packed(packed), qo.unpack_int32_to_int4(packed)


def work(case):
    size = {"fp32": 4, "fp16": 2, "bf16": 2}
    if case["kind"] in ("quant", "dequant"):
        t, f = case["tokens"], case["features"]
        if case["kind"] == "dequant":
            return {"bytes": t * f * (0.5 if case["packed"] else 1) + t * size[case["dtype"]] + t * f * 4,
                    "flops": t * f}
        m, n = qo.get_decompose_dim(f)
        es = size[case["dtype"]]
        return {"bytes": t * f * (es + (0.5 if case["pack"] else 1)) + 4 * t + (m * m + n * n) * es,
                "flops": 2 * t * f * (m + n)}
    n, k = case["n"], case["k"]
    if case["kind"] == "weight":
        return {"bytes": 3 * n * k, "flops": 0}
    m = case["m"]
    if case["kind"] == "gemm":
        return {"bytes": (m + n) * k / 2 + 2 * (m + n) + m * n * size[case["out"]], "flops": 2 * m * n * k}
    a, b = qo.get_decompose_dim(k)
    es = size[case["dtype"]]
    return {"bytes": m * k * es + (a * a + b * b) * es + n * k / 2 + 2 * n + (n * es if case["bias"] else 0) + m * n * es,
            "flops": 2 * m * n * k + 2 * m * k * (a + b)}


def tolerance(case):
    """About four times what a float32 computation with its sums in another order showed over these ranges."""
    kind = case["kind"]
    if kind in ("dequant", "weight"):
        return "exact"   # one float32 product of two exact values; bytes
    if kind == "gemm":
        # the integer sums are exact: the order of the two scale products is all that can
        # differ, by one unit of the output type (bf16: 6e-3 of a value), seldom
        return {"rel": 1e-6, "max": 1e-6} if case["out"] == "fp32" else {"rel": 2e-5, "max": 3e-2}
    if kind == "linear":
        return {"rel": 8e-3, "max": 0.6}   # a code that rounds the other way changes a row of outputs
    # Whole values are codes, or words of eight: ties that round the other way, at least one of them
    # in a small call. Scales are held in the input type: one unit of it, which a token in thousands shows.
    one = 32.0 / (case["tokens"] * case["features"])
    if case["dtype"] == "fp32":
        return {"rel": 5e-7, "max": 2e-6, "differ": min(1e-2, max(1.2e-5, one))}
    unit = 2.0 ** -10 if case["dtype"] == "fp16" else 2.0 ** -7
    return {"rel": unit, "max": 2 * unit, "differ": min(1e-2, max(1e-3, one))}


def _codes(words):
    """int32 [rows, W] -> the codes in [-8, 7], float64 [rows, 8 W]."""
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device=words.device)
    return (((words.unsqueeze(-1) >> shifts) & 15) - 8).reshape(words.shape[0], -1).double()


def _pack(codes):
    rows, feats = codes.shape
    nib = (codes.to(torch.int64) + 8).view(rows, feats // 8, 8)
    words = (nib << torch.arange(0, 32, 4, device=codes.device)).sum(2)
    return torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)


def _quantize(x, left, right, clip):
    """Codes (float64 whole numbers) and scales of Y = L^T X R, in 64 bits throughout."""
    t, (m, n) = x.shape[0], (left.shape[0], right.shape[0])
    z = (x.double().reshape(t * m, n) @ right.double()).view(t, m, n)
    y = (z.transpose(1, 2).reshape(t * n, m) @ left.double()).view(t, n, m).transpose(1, 2).reshape(t, m * n)
    scale = (torch.maximum((y.amin(1) * clip).abs(), y.amax(1) * clip) / 7.0).clamp(min=1e-8)
    return torch.round(y / scale[:, None]).clamp(-8, 7), scale


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "quant":
        q, scale = _quantize(s["x"], s["left"], s["right"], case["clip"])
        return (_pack(q) if case["pack"] else q.to(torch.int8)), scale
    if kind == "gemm":
        acc = _codes(s["a"]) @ _codes(s["b"].t()).t().contiguous()
        return acc * s["sa"].double()[:, None] * s["sb"].double()[None, :]
    if kind == "linear":
        q, scale = _quantize(s["x"], s["left"], s["right"], case["clip"])
        out = (q @ _codes(s["w"]).t().contiguous()) * scale[:, None] * s["sw"].double()[None, :]
        return out if s["bias"] is None else out + s["bias"].double()
    if kind == "dequant":
        q = _codes(s["codes"]) if case["packed"] else s["codes"].double()
        return q * s["scales"].double()[:, None]
    packed = _pack(s["codes"])
    return packed, packed.t().contiguous(), s["codes"]
