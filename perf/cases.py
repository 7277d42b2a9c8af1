"""Performance cases of the block-scaled (MX) matmul path: what a user's program has it do, through the public
Python entry points, over the sizes it does it at.

A case is a dict of plain values; ``kind`` names the entry point:

  quantize  ``block_quantize`` of an activation or weight matrix (the encode direction)
  linear    a quantised linear layer: bf16 activations -> ``block_quantize`` -> ``block_scaled_matmul`` with weights
            that were quantised when the model was loaded (decode at few rows, prefill at many); bf16 out
  gemm      ``block_scaled_matmul`` of two operands that are quantised already, plain 2-D scales
  dropin    ``cutile_block_scaled_matmul`` with ``swizzle_32_4_4`` scales, fp32 out (the sample's signature)
  mma       ``mma_scaled``: batched products with an fp32 accumulator
  list      ``grouped_block_scaled_matmul``: many small independent products in one call
  moe       ``block_quantize`` -> ``cutile_moe_scaled``: a whole mixture-of-experts feed-forward layer

Sizes are those of the benchmark and the tests (4096 / 8192 / 14336 / 28672 layers, 8 experts of 14336, top-2, the
4096^3 and 8192^3 products) and generic ones around them.
"""
import math
import pathlib
import random
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "cutile-python_amd"))

import cutile_amd as ct  # noqa: E402

FMT = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2, "e2m1": "e2m1"}
BITS = {"e4m3": 8, "e5m2": 8, "e2m1": 4}
SRC = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
OUT = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # encoding a large activation or weight matrix
        {"name": "quantize_8192_bf16_e4m3", "kind": "quantize", "rows": 8192, "K": 8192, "src": "bf16", "fmt": "e4m3",
         "mode": "floor"},
        # one sequence being decoded, attention-sized projection: the smallest call, latency and launches count
        {"name": "decode_m1_fp4", "kind": "linear", "M": 1, "N": 4096, "K": 4096, "w": "e2m1"},
        # a batch of 32 sequences being decoded, gate+up projection with FP4 weights
        {"name": "decode_m32_fp4", "kind": "linear", "M": 32, "N": 28672, "K": 8192, "w": "e2m1"},
        # a batch of 24, down projection (long K, few columns) with FP8 weights
        {"name": "decode_m24_fp8_down", "kind": "linear", "M": 24, "N": 4096, "K": 14336, "w": "e4m3"},
        # a prompt of ragged length
        {"name": "prefill_m1531_fp8", "kind": "linear", "M": 1531, "N": 14336, "K": 4096, "w": "e4m3"},
        # the benchmark's large square products
        {"name": "gemm_mxfp8_8192", "kind": "gemm", "M": 8192, "N": 8192, "K": 8192, "a": "e4m3", "b": "e4m3",
         "out": "bf16"},
        {"name": "gemm_mxfp4_8192", "kind": "gemm", "M": 8192, "N": 8192, "K": 8192, "a": "e2m1", "b": "e2m1",
         "out": "bf16"},
        # the sample's own problem, scales in the swizzled form
        {"name": "dropin_4096_swizzled", "kind": "dropin", "M": 4096, "N": 4096, "K": 4096},
        # small batched products with an accumulator, sizes that fill no tile
        {"name": "mma_scaled_batch6_e5m2", "kind": "mma", "batch": 6, "M": 200, "N": 328, "K": 992, "fmt": "e5m2"},
        # a list of small and medium problems of different sizes
        {"name": "list_24", "kind": "list", "count": 24, "shapes": 7, "lo": 96, "hi": 1536, "fmt": "e4m3",
         "out": "bf16"},
        # a mixture-of-experts layer over a full prompt batch: the largest case
        {"name": "moe_prefill_4096", "kind": "moe", "tokens": 4096, "H": 4096, "F": 14336, "E": 8, "topk": 2,
         "w": "e4m3"},
        # the same layer with FP4 weights while a batch is being decoded: every expert gets a few rows
        {"name": "moe_decode_48_fp4", "kind": "moe", "tokens": 48, "H": 4096, "F": 14336, "E": 8, "topk": 2,
         "w": "e2m1"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_mult(rng, lo, hi, m):
    return max(lo, _log(rng, lo, hi) // m * m)


def draw(rng):
    """One more case: any of the kinds, sizes spread over the logarithm of their range, ragged ones among them."""
    kind = rng.choice(["quantize", "linear", "linear", "linear", "gemm", "gemm", "dropin", "mma", "list", "moe", "moe"])
    if kind == "quantize":
        return {"kind": kind, "rows": _log(rng, 1, 8192), "K": _log_mult(rng, 512, 8192, rng.choice([32, 512])),
                "src": rng.choice(["bf16", "bf16", "f32", "f16"]), "fmt": rng.choice(["e4m3", "e4m3", "e2m1", "e5m2"]),
                "mode": rng.choice(["floor", "ceil"])}
    if kind == "linear":
        # weights are wide and aligned as a model's are; the row count is whatever the batch is
        return {"kind": kind, "M": _log(rng, 1, 4096), "N": _log_mult(rng, 1024, 28672, rng.choice([16, 256])),
                "K": _log_mult(rng, 1024, 14336, rng.choice([128, 512])), "w": rng.choice(["e2m1", "e4m3"])}
    if kind == "gemm":
        a, b = rng.choice([("e4m3", "e4m3"), ("e4m3", "e4m3"), ("e2m1", "e2m1"), ("e4m3", "e2m1"), ("e5m2", "e5m2")])
        step = rng.choice([1, 128])
        return {"kind": kind, "M": _log_mult(rng, 128, 8192, step), "N": _log_mult(rng, 128, 8192, step),
                "K": _log_mult(rng, 256, 8192, rng.choice([32, 512])), "a": a, "b": b, "out": rng.choice(["bf16", "f32"])}
    if kind == "dropin":
        return {"kind": kind, "M": _log_mult(rng, 256, 8192, 128), "N": _log_mult(rng, 256, 8192, 128),
                "K": _log_mult(rng, 256, 8192, 128)}
    if kind == "mma":
        return {"kind": kind, "batch": rng.randint(1, 8), "M": _log(rng, 16, 512), "N": _log(rng, 16, 512),
                "K": _log_mult(rng, 128, 2048, 32), "fmt": rng.choice(["e4m3", "e5m2", "e2m1"])}
    if kind == "list":
        return {"kind": kind, "count": rng.randint(4, 48), "shapes": rng.randrange(1 << 20), "lo": 32, "hi": 1536,
                "fmt": rng.choice(["e4m3", "e4m3", "e2m1"]), "out": rng.choice(["bf16", "f32"])}
    # mixtures from few wide to many narrow experts, with at most the listed layer's weights and products
    E, F = rng.choice([(8, 14336), (8, 7168), (16, 4096), (32, 2048), (64, 1024)])
    topk = rng.choice([1, 2] if E == 8 else [2, 4])
    return {"kind": kind, "tokens": _log(rng, 1, 8192 // topk), "H": _log_mult(rng, 1024, 4096, 512), "F": F, "E": E,
            "topk": topk, "w": rng.choice(["e4m3", "e2m1"])}


def _list_shapes(case):
    r = random.Random(case["shapes"])
    lo, hi = case["lo"], case["hi"]
    return [(_log(r, lo, hi), _log(r, lo, hi), max(32, _log(r, lo, hi) // 32 * 32)) for _ in range(case["count"])]


class _Maker:
    """Random operands on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, shape, std=1.0, dtype=torch.float32):
        return torch.empty(shape, device=self.dev, dtype=dtype).normal_(0.0, std, generator=self.g)

    def quantized(self, rows, K, fmt, std=1.0):
        """(elements, scales) of a random (rows, K) matrix; E2M1 operands are spread over the format's range."""
        if fmt == "e2m1" and std == 1.0:
            x = torch.empty((rows, K), device=self.dev).uniform_(-6.0, 6.0, generator=self.g)
        else:
            x = self.normal((rows, K), std)
        return ct.block_quantize(x, 32, FMT[fmt], scale_mode="floor")


def prepare(case, seed):
    m = _Maker(seed)
    kind = case["kind"]
    s = {"case": dict(case)}
    if kind == "quantize":
        s["x"] = m.normal((case["rows"], case["K"]), 1.0, SRC[case["src"]])
    elif kind == "linear":
        s["x"] = m.normal((case["M"], case["K"]), 1.0, torch.bfloat16)
        w, ws = m.quantized(case["N"], case["K"], case["w"], 0.02)
        # the skinny-M kernel for FP4 weights reads plain scales; everything else takes them packed at load time
        skinny = case["w"] == "e2m1" and case["M"] <= 64
        s["w"], s["ws"] = w.T, ws.T if skinny else ct.pack_scales(ws, operand="b")
    elif kind == "gemm":
        s["a"], s["as"] = m.quantized(case["M"], case["K"], case["a"])
        b, bs = m.quantized(case["N"], case["K"], case["b"])
        s["b"], s["bs"] = b.T, bs.T
    elif kind == "dropin":
        s["a"], a_s = m.quantized(case["M"], case["K"], "e4m3")
        b, b_s = m.quantized(case["N"], case["K"], "e4m3")
        s["as"], s["b"], s["bs"] = ct.swizzle_32_4_4(a_s), b.T, ct.swizzle_32_4_4(b_s)
    elif kind == "mma":
        n, M, N, K = case["batch"], case["M"], case["N"], case["K"]
        a, a_s = m.quantized(n * M, K, case["fmt"])
        b, b_s = m.quantized(n * N, K, case["fmt"])
        s["a"], s["as"] = a.view(n, M, -1), a_s.view(n, M, -1)
        s["b"], s["bs"] = b.view(n, N, -1).transpose(1, 2), b_s.view(n, N, -1).transpose(1, 2)
        s["acc"] = m.normal((n, M, N))
    elif kind == "list":
        view = torch.float4_e2m1fn_x2 if case["fmt"] == "e2m1" else FMT[case["fmt"]]
        s["a"], s["as"], s["b"], s["bs"] = [], [], [], []
        for M, N, K in _list_shapes(case):
            a, a_s = m.quantized(M, K, case["fmt"])
            b, b_s = m.quantized(N, K, case["fmt"])
            s["a"].append(a.view(view))
            s["as"].append(a_s)
            s["b"].append(b.view(view).T)
            s["bs"].append(b_s.T)
    else:
        T, H, F, E, k = (case[n] for n in ("tokens", "H", "F", "E", "topk"))
        s["x"] = m.normal((T, H), 1.0, torch.bfloat16)
        for name, rows, K in (("w1", 2 * F, H), ("w2", H, F)):
            w, ws = m.quantized(E * rows, K, case["w"], 0.02)
            s[name] = w.view(E, rows, -1)
            s[name + "s"] = ct.pack_scales(ws.view(E, rows, -1), operand="b")
        logits = m.normal((T, E))
        top, s["ids"] = logits.topk(k, dim=1)
        s["weights"] = torch.softmax(top, dim=1)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "quantize":
        q, sc = ct.block_quantize(s["x"], 32, FMT[case["fmt"]], scale_mode=case["mode"])
        return q.view(torch.uint8), sc.view(torch.uint8)
    if kind == "linear":
        q, sc = ct.block_quantize(s["x"], 32, torch.float8_e4m3fn, scale_mode="floor")
        return ct.block_scaled_matmul(q, sc, s["w"], s["ws"], b_format=case["w"], out_dtype=torch.bfloat16)
    if kind == "gemm":
        return ct.block_scaled_matmul(s["a"], s["as"], s["b"], s["bs"], a_format=case["a"], b_format=case["b"],
                                      out_dtype=OUT[case["out"]])
    if kind == "dropin":
        return ct.cutile_block_scaled_matmul(s["a"], s["as"], s["b"], s["bs"])
    if kind == "mma":
        return ct.mma_scaled(s["a"], s["as"], s["b"], s["bs"], s["acc"], x_format=case["fmt"], y_format=case["fmt"])
    if kind == "list":
        return ct.grouped_block_scaled_matmul(s["a"], s["as"], s["b"], s["bs"], out_dtype=OUT[case["out"]])
    q, sc = ct.block_quantize(s["x"], 32, torch.float8_e4m3fn, scale_mode="floor")
    return ct.cutile_moe_scaled(q, sc, s["w1"], s["w1s"], s["w2"], s["w2s"], s["weights"], s["ids"],
                                w_format=case["w"])


def _operand(rows, K, fmt):
    """Bytes of an MX operand: elements and one scale per 32 of them."""
    return rows * K * BITS[fmt] / 8 + rows * K / 32


def work(case):
    kind = case["kind"]
    if kind == "quantize":
        n = case["rows"] * case["K"]
        return {"bytes": n * (4 if case["src"] == "f32" else 2) + _operand(case["rows"], case["K"], case["fmt"]),
                "flops": 2 * n}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * M * K + _operand(N, K, case["w"]) + 2 * M * N, "flops": 2 * M * N * K}
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _operand(M, K, case["a"]) + _operand(N, K, case["b"]) + M * N * (2 if case["out"] == "bf16" else 4),
                "flops": 2 * M * N * K}
    if kind == "dropin":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _operand(M, K, "e4m3") + _operand(N, K, "e4m3") + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "mma":
        n, M, N, K = case["batch"], case["M"], case["N"], case["K"]
        return {"bytes": _operand(n * M, K, case["fmt"]) + _operand(n * N, K, case["fmt"]) + 8 * n * M * N,
                "flops": 2 * n * M * N * K}
    if kind == "list":
        c = 2 if case["out"] == "bf16" else 4
        b = f = 0
        for M, N, K in _list_shapes(case):
            b += _operand(M, K, case["fmt"]) + _operand(N, K, case["fmt"]) + c * M * N
            f += 2 * M * N * K
        return {"bytes": b, "flops": f}
    T, H, F, E, k = (case[n] for n in ("tokens", "H", "F", "E", "topk"))
    touched = E * (1.0 - (1.0 - k / E) ** T)   # experts that at least one token is expected to go to
    return {"bytes": touched * (_operand(2 * F, H, case["w"]) + _operand(H, F, case["w"])) + 4 * T * H,
            "flops": 2 * T * k * 3 * F * H}


def tolerance(case):
    """bf16 outputs: two correct results differ by their own rounding (2^-9 of the value at most, 0.0024 in the mean for
    two independent ones).  fp32 outputs: order of summation and the matrix instruction's own rounding.  The MoE
    layer rounds its intermediate activation to bf16 and then to E4M3, where a last-bit difference can move a value
    by one step."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "moe":
        return {"rel": 1e-2}
    if kind in ("dropin", "mma") or case.get("out") == "f32":
        return {"rel": 3e-5}
    return {"rel": 4e-3}
