"""The fp32 plane kernels (csrc/gemm_f32_x6.hip): tile and K edges in every
layout at any 4-byte alignment, values their bf16 planes do not hold, and an
error against 64 bits no larger than the fp32 MFMA kernel's."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

pytestmark = pytest.mark.gpu

PLANES = [v["name"] for v in _lib.variants() if v["name"].endswith("_x6")]
# around the tiles (64, 128, 256), the K steps (16, 32) and fewer K than a step
SHAPES = [(1, 1, 1), (64, 16, 64), (65, 15, 63), (127, 17, 129), (128, 32, 128), (129, 33, 257), (257, 1, 130),
          (256, 48, 256), (255, 63, 300), (300, 1099, 70)]


def view(x, col, gap, shift):
    """Device tensor of x, row- or column-major, rows `gap` elements longer
    than x's and the first one `shift` elements into its allocation."""
    rows, cols = (x.shape[1], x.shape[0]) if col else x.shape
    flat = torch.full((shift + rows * (cols + gap),), float("nan"), dtype=torch.float32, device="cuda")
    v = flat.as_strided((rows, cols), (cols + gap, 1), shift)
    v.copy_(torch.from_numpy(np.ascontiguousarray(x.T if col else x)))
    return v.t() if col else v


def run(x1, x2, cfg):
    out = ext.matrix_mul(x1, x2, cfg)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("name", PLANES)
def test_edges_layouts_alignment(name):
    splits = (1, 3) if ext.tile_can_split(_lib.variants()[_lib.variant_id(name)]) else (1,)
    for i, (m, k, n) in enumerate(SHAPES):
        a, b = O.normal((m, k), 40 + 2 * i), O.normal((k, n), 41 + 2 * i)
        ref = O.matmul_f64(a, b)
        for layout in range(4):
            gap, shift = ((0, 0), (1, 1), (5, 2), (8, 3))[(i + layout) % 4]
            x1, x2 = view(a, layout & 1, gap, shift), view(b, layout & 2, gap, 3 - shift)
            for s in splits:
                print(name, (m, k, n), "layout", layout, "gap", gap, "split", s, flush=True)
                # up to 6 K / 16 = 413 roundings of the sum: sqrt(413) 2^-25, and twice that
                assert O.rel_l2(run(x1, x2, (name, s)), ref) <= 1.2e-6


@pytest.mark.parametrize("name", PLANES)
def test_magnitudes_infinities_nan(name):
    m, k, n = 150, 130, 140
    a, b = O.normal((m, k), 1), O.normal((k, n), 2)
    plain = ("gemm_f32_64x64x16_w2x2", 1)
    # tiny and huge operands, whose planes or plane products underflow or overflow
    for sa, sb in [(1e-15, 1), (1e-20, 1e-12), (1e-25, 1e25), (1e-36, 1e30), (1e36, 1e-36), (1e-10, 1e-26), (0, 1)]:
        x, y = (a * np.float32(sa)).astype(np.float32), (b * np.float32(sb)).astype(np.float32)
        got = run(view(x, 0, 0, 0), view(y, 0, 0, 0), (name, 1))
        ref = O.matmul_f64(x, y)
        print(name, "scales", sa, sb, flush=True)
        assert np.array_equal(got, ref) if sa == 0 else O.rel_l2(got, ref) <= 1e-6
    # rows of very different magnitudes, each against its own row of the reference
    x = (a * np.logspace(-30, 30, m)[:, None]).astype(np.float32)
    got, ref = run(view(x, 0, 0, 0), view(b, 0, 0, 0), (name, 1)).astype(np.float64), O.matmul_f64(x, b)
    assert (np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)).max() <= 2e-6
    for bad in (np.inf, -np.inf, np.nan, 3.4e38):
        x = a.copy()
        x[3, 5] = x[149, 129] = bad
        got, want = run(view(x, 0, 0, 0), view(b, 0, 0, 0), (name, 1)), run(view(x, 0, 0, 0), view(b, 0, 0, 0), plain)
        print(name, "value", bad, flush=True)
        fin = np.isfinite(want)
        np.testing.assert_array_equal(got[~fin], want[~fin])
        assert O.rel_l2(got[fin], want[fin]) <= 1e-6


@pytest.mark.parametrize("name", PLANES)
def test_error_no_larger_than_the_fp32_mfma_kernel(name):
    for k in (64, 512, 4096):
        a, b = O.normal((256, k), 7), O.normal((k, 256), 8)
        ref = O.matmul_f64(a, b)
        x1, x2 = view(a, 0, 0, 0), view(b, 0, 0, 0)
        err, plain = (O.rel_l2(run(x1, x2, (v, 1)), ref) for v in (name, "gemm_f32_128x128x16_w2x2"))
        print(name, k, err, plain, flush=True)
        assert err <= plain
