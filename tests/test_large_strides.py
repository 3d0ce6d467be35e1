"""Row strides on either side of what the in-place tile kernels' 32-bit offsets
take: the fp32 plane kernels (csrc/gemm_f32_x6.hip) hand larger ones to the
register-staged kernel of the same tile, the bf16 kernels of any alignment
(csrc/gemm_bf16_any.hip) to the generic one."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

pytestmark = pytest.mark.gpu

LIMIT = (1 << 31) - 4096  # bytes of a K step's offsets
BY_NAME = {v["name"]: v for v in _lib.variants()}
PLANES = [n for n in BY_NAME if n.endswith("_x6")]
ANY = [n for n in BY_NAME if n.endswith("_any")]


def spread(t, ld):
    """t (rows, cols) on the device with a row stride of ld elements."""
    flat = torch.empty((t.shape[0] - 1) * ld + t.shape[1], dtype=t.dtype, device="cuda")
    v = flat.as_strided(t.shape, (ld, 1))
    v.copy_(t)
    return v


@pytest.mark.parametrize("name", PLANES)
@pytest.mark.parametrize("operand", ["x1 rows", "x1 columns", "x2 rows", "x2 columns"])
def test_planes(name, operand):
    v = BY_NAME[name]
    m, k, n = v["bm"] + 1, 37, v["bn"] + 2
    a, b = O.normal((m, k), 70), O.normal((k, n), 71)
    ref = O.matmul_f64(a, b)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    # rows of the strided view that one K step takes, and what it holds
    step, t = {"x1 rows": (v["bm"], ta), "x1 columns": (v["bk"], ta.t()),
               "x2 rows": (v["bk"], tb), "x2 columns": (v["bn"], tb.t())}[operand]
    for ld in (LIMIT // 4 // step - 1, -(-LIMIT // 4 // step)):  # the last that fits, the first that does not
        w = spread(t.contiguous(), ld)
        x1 = w if operand == "x1 rows" else w.t() if operand == "x1 columns" else ta
        x2 = w if operand == "x2 rows" else w.t() if operand == "x2 columns" else tb
        for s in (1, 2) if ext.tile_can_split(v) else (1,):
            print(name, operand, "stride", ld, "split", s, flush=True)
            got = ext.matrix_mul(x1, x2, (name, s)).cpu().numpy()
            # at most 37 roundings of the sum: sqrt(37) 2^-25, and twice that
            assert O.rel_l2(got, ref) <= 3.7e-7
        del w, x1, x2


@pytest.mark.parametrize("name", ANY + ["gemm_bf16_128x128x64_r4_m16"])
@pytest.mark.parametrize("operand", ["x1 rows", "x1 columns", "x2 rows", "x2 columns"])
def test_any_alignment(name, operand):
    m, k, n = 129, 75, 67
    a, b = O.bf16_round(O.normal((m, k), 72)), O.bf16_round(O.normal((k, n), 73))
    ref = O.matmul_bf16_f64(a, b)
    dev = lambda h: torch.from_numpy(np.ascontiguousarray(h).view(np.int16)).cuda().view(torch.bfloat16)
    ta, tb = dev(a), dev(b)
    t = {"x1 rows": ta, "x1 columns": ta.t(), "x2 rows": tb, "x2 columns": tb.t()}[operand]
    top = LIMIT // 256  # 128 rows of 2 bytes
    for ld in (top - 1 - top % 2, top + 1 + top % 2):  # odd: rows of any alignment
        w = spread(t.contiguous(), ld)
        x1 = w if operand == "x1 rows" else w.t() if operand == "x1 columns" else ta
        x2 = w if operand == "x2 rows" else w.t() if operand == "x2 columns" else tb
        for s in (1, 2):
            print(name, operand, "stride", ld, "split", s, flush=True)
            got = ext.matrix_mul(x1, x2, (name, s)).cpu().numpy()
            # sums of 75 exact products, at most one rounding per 16
            assert O.rel_l2(got, ref) <= 5e-7
        del w, x1, x2
