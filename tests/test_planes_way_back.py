"""Sums of the fp32 plane kernels (csrc/gemm_f32_x6.hip) that are not finite
are multiplied again on the fp32 MFMAs: eight k a step, four steps in flight,
every remainder of K, each layout, and only the row blocks that hold one."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

pytestmark = pytest.mark.gpu

PLANES = [v["name"] for v in _lib.variants() if v["name"].endswith("_x6")]


def view(x, col, gap):
    """x on the device, row- or column-major, NaN between its rows."""
    rows, cols = (x.shape[1], x.shape[0]) if col else x.shape
    flat = torch.full((rows * (cols + gap) + 1,), float("nan"), device="cuda")
    v = flat.as_strided((rows, cols), (cols + gap, 1), 1)
    v.copy_(torch.from_numpy(np.ascontiguousarray(x.T if col else x)))
    return v.t() if col else v


@pytest.mark.parametrize("name", PLANES)
def test_remainders_and_layouts(name):
    """Integers times 2^50 each: exact in fp32, sums above 2^96."""
    splits = (1, 3) if ext.tile_can_split(_lib.variants()[_lib.variant_id(name)]) else (1,)
    for i, k in enumerate((1, 7, 8, 9, 31, 32, 33, 39, 64, 203)):
        m, n = (130, 67) if i % 2 else (65, 257)
        a, b = (np.ldexp(O.small_ints(s, 60 + 2 * i + j, -8, 8).astype(np.float32), 50)
                for j, s in enumerate(((m, k), (k, n))))
        want = a.astype(np.float64) @ b.astype(np.float64)
        for layout in range(4):
            for s in splits:
                print(name, (m, k, n), "layout", layout, "split", s, flush=True)
                got = ext.matrix_mul(view(a, layout & 1, i % 3), view(b, layout & 2, (i + 1) % 3), (name, s))
                assert (got.cpu().numpy() == want).all()


@pytest.mark.parametrize("name", PLANES)
def test_one_infinity(name):
    """One infinity in each operand: its row and its column are infinities and
    NaN as in the fp32 kernels, everything else is what it is without them."""
    m, k, n = 300, 100, 270
    a, b = O.normal((m, k), 8), O.normal((k, n), 9)
    a2, b2 = a.copy(), b.copy()
    a2[137, 41], b2[77, 200] = np.inf, -np.inf
    want = a2.astype(np.float64) @ b2.astype(np.float64)
    for layout in range(4):
        got = ext.matrix_mul(view(a2, layout & 1, 1), view(b2, layout & 2, 2), (name, 1)).cpu().numpy()
        fin = np.isfinite(want)
        assert fin.sum() == (m - 1) * (n - 1)
        np.testing.assert_array_equal(got[~fin], want[~fin].astype(np.float32))
        # up to 100 roundings of the sum: sqrt(100) 2^-25, and twice that
        assert O.rel_l2(got[fin], want[fin]) <= 6e-7
