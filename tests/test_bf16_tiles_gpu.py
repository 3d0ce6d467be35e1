"""The bf16 kernels for outputs of few tiles: direct-to-LDS tiles of 64 and
128 on four waves, and the tiles that read any element alignment
(csrc/gemm_bf16_any.hip), at the edges of tiles, K steps and 16-byte groups in
every layout."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

pytestmark = pytest.mark.gpu

ANY = [v["name"] for v in _lib.variants() if v["name"].endswith("_any")]
SMALL = ["gemm_bf16_64x64x64_r4_m16", "gemm_bf16_128x64x64_r3_m16", "gemm_bf16_64x128x64_r3_m16",
         "gemm_bf16_128x128x64_r2w4_m16"]
# sums of K <= 1100 products in fp32, at most one rounding per 16: sqrt(70) 2^-25 and twice that
TOL = 5e-7


def view(h, col, gap, shift):
    """bf16 device view of the bit patterns h, row- or column-major, rows `gap`
    elements longer (NaN between them), `shift` elements into its allocation."""
    rows, cols = (h.shape[1], h.shape[0]) if col else h.shape
    flat = torch.full((shift + (rows - 1) * (cols + gap) + cols,), float("nan"), dtype=torch.bfloat16, device="cuda")
    v = flat.as_strided((rows, cols), (cols + gap, 1), shift)
    v.copy_(torch.from_numpy(np.ascontiguousarray(h.T if col else h).view(np.int16)).cuda().view(torch.bfloat16))
    return v.t() if col else v


def check(name, m, k, n, seed, layout, gap, shift, splits):
    a, b = O.bf16_round(O.normal((m, k), seed)), O.bf16_round(O.normal((k, n), seed + 1))
    ref = O.matmul_bf16_f64(a, b)
    x1, x2 = view(a, layout & 1, gap, shift), view(b, layout & 2, gap, shift)
    for s in splits:
        print(name, (m, k, n), "layout", layout, "gap", gap, "shift", shift, "split", s, flush=True)
        out = ext.matrix_mul(x1, x2, (name, s))
        torch.cuda.synchronize()
        assert O.rel_l2(out.cpu().numpy(), ref) <= TOL


# K below 8 (the generic kernel), one straddling chunk, around the 64-deep step;
# single rows and columns, odd extents, tile edges
@pytest.mark.parametrize("name", ANY)
def test_any_alignment(name):
    for i, (m, k, n) in enumerate([(1, 8, 2), (2, 7, 3), (3, 9, 1), (65, 63, 129), (64, 65, 127), (129, 71, 63),
                                   (127, 128, 65), (130, 257, 131), (63, 1099, 64)]):
        for layout in range(4):
            gap, shift = ((0, 0), (1, 0), (0, 1), (3, 5))[(i + layout) % 4]
            check(name, m, k, n, 60 + 2 * i, layout, gap, shift, (1, 3))


@pytest.mark.parametrize("name", SMALL)
def test_small_tiles(name):
    for i, (m, k, n) in enumerate([(8, 8, 8), (64, 64, 64), (72, 200, 136), (128, 72, 56), (136, 1088, 120)]):
        for layout in range(4):
            check(name, m, k, n, 90 + 2 * i, layout, 8 * (i % 2), 0, (1, 2))
            # operands it does not take in place: rows at odd offsets
            check(name, m, k, n, 90 + 2 * i, layout, 1, 1, (1, 2))


def test_rows_apart_by_an_odd_stride():
    """The picked config (by extents, which are aligned) on a column slice whose
    row stride is odd."""
    for m, k, n in [(300, 256, 512), (2048, 128, 2048)]:
        a, b = O.bf16_round(O.normal((m, k), 3)), O.bf16_round(O.normal((k, n), 4))
        out = ext.matrix_mul(view(a, 0, 5, 1), view(b, 0, 0, 0))
        torch.cuda.synchronize()
        assert O.rel_l2(out.cpu().numpy(), O.matmul_bf16_f64(a, b)) <= TOL
