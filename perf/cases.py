"""What the speed of this package is judged by: calls of `tilec.ext.matrix_mul`
and `tilec.ext.sum` over the range of sizes, layouts and types that they are
used with, each with its inputs, its algorithmic work, the tolerance of its
outputs and a 64-bit reference.

Three kinds of case ("op"):
  mm      out = x1 @ x2.  "layout" says how the operands lie in memory:
          "nn" both row-major; "nt" x2 the transposed view of a row-major
          weight [N, K] (x @ W.T: a linear layer's forward pass, prefill and
          decode); "tn" x1 a transposed view (dy.T @ x: a weight gradient).
          "gap" > 0: x1 is a column slice of a wider matrix with that many
          columns more (one part of a fused projection's output).
  linear  one training step's products of a linear layer: the forward
          x @ W.T, the input gradient dy @ W, the weight gradient dy.T @ x
          and the bias gradient sum(dy, axis=0).
  sum     row sums (axis 1) or column sums (axis 0).
"""

import math

import torch

import tilec

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _mm(name, dtype, layout, M, K, N, gap=0):
    return {"name": name, "op": "mm", "dtype": dtype, "layout": layout, "M": M, "K": K, "N": N, "gap": gap}


def _linear(name, dtype, T, K, N):
    return {"name": name, "op": "linear", "dtype": dtype, "T": T, "K": K, "N": N}


def _sum(name, dtype, axis, R, C):
    return {"name": name, "op": "sum", "dtype": dtype, "axis": axis, "R": R, "C": C}


def listed():
    return [
        # The smallest call: a small ragged product, all latency and host work.
        _mm("f32_tiny", "f32", "nn", 65, 17, 63),
        # The README's example product.
        _mm("f32_readme", "f32", "nn", 512, 4096, 64),
        # A single row against a 64 MiB row-major matrix (the GEMV workload).
        _mm("f32_gemv", "f32", "nn", 1, 4096, 4096),
        # A ragged product: every tile edge out of bounds, odd row strides.
        _mm("f32_ragged", "f32", "nn", 1000, 4097, 3001),
        # The headline: a large square fp32 product.
        _mm("f32_square", "f32", "nn", 4096, 4096, 4096),
        # Decoding 16 sequences at a time through a bf16 linear layer.
        _mm("bf16_decode", "bf16", "nt", 16, 4096, 4096),
        # A short prompt (or a large decode batch) through a bf16 linear layer.
        _mm("bf16_prefill", "bf16", "nt", 128, 4096, 4096),
        # Operand rows that are not whole 16-byte groups.
        _mm("bf16_ragged", "bf16", "nn", 1359, 4447, 1009),
        # The largest product: bf16, fp32 accumulate.
        _mm("bf16_square", "bf16", "nn", 8192, 8192, 8192),
        # Training steps of a linear layer: mixed precision, and a smaller fp32
        # one whose output (1000 classes) is no multiple of a tile.
        _linear("bf16_step", "bf16", 2048, 4096, 4096),
        _linear("f32_step", "f32", 512, 2048, 1000),
        # Row sums of a 64 MiB matrix.
        _sum("f32_row_sum", "f32", 1, 4096, 4096),
    ]


# Limits of a drawn case, all below the largest listed one's cost.
MAX_ELEMS = 1 << 25
MAX_FLOPS = {"f32": 1 << 36, "bf16": 1 << 38}


def _size(rng, lo, hi):
    """A size log-uniform in [lo, hi]; half of those above 64 are multiples of
    64, as model widths are, the rest any whole number."""
    v = max(lo, min(hi, round(2 ** rng.uniform(math.log2(lo), math.log2(hi)))))
    return v // 64 * 64 if v > 64 and rng.random() < 0.5 else v


def draw(rng):
    while True:
        dtype = rng.choice(("f32", "bf16"))
        kind = rng.random()
        if kind < 0.15:
            c = {"op": "sum", "dtype": dtype, "axis": rng.choice((0, 1)), "R": _size(rng, 8, 65536),
                 "C": _size(rng, 8, 65536)}
            if c["R"] * c["C"] <= MAX_ELEMS:
                return c
        elif kind < 0.3:
            c = {"op": "linear", "dtype": dtype, "T": _size(rng, 16, 4096), "K": _size(rng, 64, 8192),
                 "N": _size(rng, 16, 8192)}
            M, K, N, flops = c["T"], c["K"], c["N"], 6 * c["T"] * c["K"] * c["N"]
            if max(M * K, K * N, M * N) <= MAX_ELEMS and flops <= MAX_FLOPS[dtype]:
                return c
        else:
            few = rng.random() < 0.3
            M = rng.randint(1, 16) if few else _size(rng, 17, 8192)
            layout = rng.choice(("nn", "nt")) if few else rng.choice(("nn", "nn", "nt", "nt", "tn"))
            K, N = _size(rng, 16, 16384), _size(rng, 16, 16384)
            gap = _size(rng, 8, 4096) if layout != "tn" and rng.random() < 0.15 else 0
            if max(M * (K + gap), K * N, M * N) <= MAX_ELEMS and 2 * M * K * N <= MAX_FLOPS[dtype]:
                return {"op": "mm", "dtype": dtype, "layout": layout, "M": M, "K": K, "N": N, "gap": gap}


def _normal(gen, dtype, rows, cols, std=1.0):
    return torch.randn(rows, cols, generator=gen, device="cuda").mul_(std).to(DTYPES[dtype])


def prepare(case, seed):
    """Inputs on the GPU: activations and gradients N(0, 1), weights
    N(0, 1 / K)."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = case["dtype"]
    if case["op"] == "sum":
        return {"case": case, "x": _normal(gen, dt, case["R"], case["C"])}
    if case["op"] == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        return {"case": case, "x": _normal(gen, dt, T, K), "w": _normal(gen, dt, N, K, 1 / math.sqrt(K)),
                "dy": _normal(gen, dt, T, N)}
    M, K, N, gap = case["M"], case["K"], case["N"], case["gap"]
    if case["layout"] == "tn":
        x1 = _normal(gen, dt, K, M).t()
    else:
        x1 = _normal(gen, dt, M, K + gap)[:, :K]
    std = 1 / math.sqrt(K)
    x2 = _normal(gen, dt, N, K, std).t() if case["layout"] == "nt" else _normal(gen, dt, K, N, std)
    return {"case": case, "x1": x1, "x2": x2}


def run(state):
    case = state["case"]
    if case["op"] == "sum":
        return tilec.ext.sum(state["x"], axis=case["axis"])
    if case["op"] == "linear":
        x, w, dy = state["x"], state["w"], state["dy"]
        return {"y": tilec.ext.matrix_mul(x, w.t()), "dx": tilec.ext.matrix_mul(dy, w),
                "dw": tilec.ext.matrix_mul(dy.t(), x), "db": tilec.ext.sum(dy, axis=0)}
    return tilec.ext.matrix_mul(state["x1"], state["x2"])


def exact(case, seed):
    """run()'s outputs in 64 bits, by torch (contiguous float64 operands)."""
    s = {k: v.double().contiguous() for k, v in prepare(case, seed).items() if k != "case"}
    if case["op"] == "sum":
        return s["x"].sum(dim=case["axis"])
    if case["op"] == "linear":
        x, w, dy = s["x"], s["w"], s["dy"]
        return {"y": torch.mm(x, w.t().contiguous()), "dx": torch.mm(dy, w),
                "dw": torch.mm(dy.t().contiguous(), x), "db": dy.sum(dim=0)}
    return torch.mm(s["x1"], s["x2"])


def work(case):
    esz = 4 if case["dtype"] == "f32" else 2
    if case["op"] == "sum":
        R, C = case["R"], case["C"]
        return {"bytes": esz * R * C + 4 * (R if case["axis"] == 1 else C), "flops": R * C}
    if case["op"] == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        return {"bytes": esz * (T * K + N * K + T * N) + 4 * (T * N + T * K + N * K + N),
                "flops": 6 * T * K * N + T * N}
    M, K, N = case["M"], case["K"], case["N"]
    return {"bytes": esz * (M * K + K * N) + 4 * M * N, "flops": 2 * M * K * N}


def tolerance(case):
    """Inputs are exact in both types (a bf16 product is exact in 32 bits) and
    everything is accumulated in 32 bits, so outputs differ by the order of
    summation, which grows as the root of its length L.  Measured against 64
    bits: 1.1e-6 at L = 4096 for fp32 products (one running sum per output);
    four times that, and never under 1e-6."""
    if case["op"] == "sum":
        L = case["C"] if case["axis"] == 1 else case["R"]
    elif case["op"] == "linear":
        L = max(case["T"], case["K"], case["N"])
    else:
        L = case["K"]
    return {"rel": max(1e-6, 4.4e-6 * math.sqrt(L / 4096))}
