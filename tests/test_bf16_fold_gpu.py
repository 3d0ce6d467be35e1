"""The four-wave bf16 tiles and the any-alignment tiles move their running sums
to a second set about every 256 k (csrc/gemm_bf16_lds.hip, gemm_bf16_any.hip)."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

pytestmark = pytest.mark.gpu

NAMES = ["gemm_bf16_64x64x64_r4_m16", "gemm_bf16_128x64x64_r3_m16", "gemm_bf16_64x128x64_r3_m16",
         "gemm_bf16_128x128x64_r2w4_m16"] + [v["name"] for v in _lib.variants() if v["name"].endswith("_any")]


def dev(h):
    return torch.from_numpy(np.ascontiguousarray(h).view(np.int16)).cuda().view(torch.bfloat16)


@pytest.mark.parametrize("name", NAMES)
def test_turns_of_the_ring(name):
    """Integers, exact in fp32: every product counted once, whatever number of
    steps is left after the last fold (and with K no multiple of a step)."""
    for i, K in enumerate((64, 192, 248, 256, 320, 384, 448, 512, 576, 768, 1016, 1024, 1031)):
        a, b = (O.small_ints(s, 1700 + 2 * i + j, -8, 8).astype(np.float32) for j, s in enumerate(((70, K), (K, 72))))
        print(name, K, flush=True)
        out = ext.matrix_mul(dev(O.bf16_round(a)), dev(O.bf16_round(b)), (name, 1))
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("name", NAMES)
def test_error_of_a_long_sum(name):
    """K = 8192 unsplit.  A rounding's relative error is 2^-24 / sqrt(3) at
    most in the mean; n additions of like terms give it sqrt(n / 2) times.  A
    fold of 384 k is at most 24 additions and 8192 k at least 22 folds: 1.2e-7
    and 1.1e-7, 1.7e-7 together (32 folds of 256 k the same).  One running sum
    of 512 additions has 5.5e-7."""
    for K in (8192, 8191):
        a, b = O.bf16_round(O.normal((128, K), 1750)), O.bf16_round(O.normal((K, 128), 1751))
        print(name, K, flush=True)
        out = ext.matrix_mul(dev(a), dev(b), (name, 1))
        torch.cuda.synchronize()
        assert O.rel_l2(out.cpu().numpy(), O.matmul_bf16_f64(a, b)) <= 2.5e-7
