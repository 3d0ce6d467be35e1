"""`tune.pick` leaves the more exact choice of the two reference models only for
a config whose sums are measured to be no less exact."""

import math
import random

import pytest
import torch

from tilec import ext, tune

# shapes (M, K, N, dtype, layout) and the configs that ran them before kernels with other orders of summation came
CASES = [
    ((512, 2048, 1000, "f32", 2), ("gemm_f32_64x64x32_w2x2_lds", 4)),
    ((64, 4096, 4096, "f32", 2), ("gemm_f32_64x64x64_w2x2_lds", 8)),
    ((96, 6144, 2048, "f32", 2), ("gemm_f32_64x64x32_w2x2_lds", 8)),
    ((106, 4032, 1728, "f32", 2), ("gemm_f32_64x64x32_w2x2_lds", 8)),
    ((4096, 1, 4096, "f32", 0), ("gemm_f32_256x256x16_w2x4", 1)),
    ((4096, 2, 4096, "f32", 0), ("gemm_f32_256x256x16_w2x4", 1)),
    ((192, 5927, 4508, "f32", 0), ("gemm_f32_64x64x16_w2x2", 16)),
    ((6912, 92, 88, "f32", 1), ("skinny_f32_w4_b1", 1)),
    ((64, 8215, 71, "f32", 2), ("direct_f32_16x64_w8", 32)),
    ((37, 704, 6912, "f32", 2), ("direct_f32_32x64_w4_db", 1)),
    ((9, 134, 12279, "bf16", 2), ("skinny_bf16_w4_b1", 2)),
    ((3, 532, 3008, "bf16", 2), ("skinny_bf16_t4_r2_w4", 1)),
    ((5, 225, 6272, "bf16", 0), ("skinny_bf16_w4_b2", 2)),
    ((1344, 4187, 2685, "bf16", 1), ("gemm_bf16_256x128x64_r3_m16_pad", 2)),
    ((128, 4096, 4096, "bf16", 2), None),
    ((1000, 4097, 3001, "f32", 0), None),
    # more exact configs of the later kernels
    ((4096, 16, 4096, "f32", 0), ("gemm_f32_256x256x16_x6", 1)),
    ((382, 117, 2954, "f32", 2), ("gemm_f32_64x64x16_d4_x6", 1)),
    ((606, 1732, 3584, "f32", 2), ("gemm_f32_128x128x16_x6", 4)),
    ((128, 4822, 1792, "f32", 2), ("gemm_f32_128x128x32_w8_x6", 16)),
    ((358, 6948, 4111, "bf16", 0), ("gemm_bf16_128x128x64_any", 4)),
    ((640, 13184, 1245, "bf16", 1), ("gemm_bf16_128x128x64_any", 4)),
]


def test_reference_choices():
    for shape, config in CASES:
        if config is not None:
            assert tune.reference(*shape) == config, shape


def test_picks_are_no_less_exact_by_the_measured_errors():
    rng = random.Random(8)
    size = lambda lo, hi: round(2 ** rng.uniform(math.log2(lo), math.log2(hi)))
    shapes = [s for s, _ in CASES] + [
        (rng.choice((size(1, 16), size(17, 4096))), size(1, 8192), size(16, 8192), dtype, rng.choice((0, 1, 2)))
        for dtype in ("f32", "bf16") for _ in range(60)]
    for s in shapes:
        config, ref = tune.pick(*s), tune.reference(*s)
        assert config in ext.hip_configs(*s)
        assert config == ref or tune.no_less_exact(config, ref, s[1]), (s, config, ref)


def test_errors_between_powers_of_two():
    """Every variant has been measured unsplit; a value between two measured
    ones lies between them."""
    for v in tune._variant_by_name():
        for k in (1, 3, 100, 5000, 16384, 100000):
            assert tune.sum_error(v, 1, k) is not None
    for name, split in (("gemm_f32_64x64x32_w2x2_lds", 4), ("direct_f32_16x64_w4_db", 6), ("gemm_bf16_64x64x64_any", 3)):
        lo, mid, hi = (tune.sum_error(name, split, k) for k in (2048, 3000, 4096))
        assert lo <= mid <= hi
    assert tune.sum_error("gemm_f32_64x64x32_w2x2_lds", 8, 4096) < tune.sum_error("gemm_f32_64x64x32_w2x2_lds", 4, 4096)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,config", CASES)
def test_picked_sums(shape, config):
    """The error of the pick against 64 bits, beside that of the reference: no
    larger but for the 5 % that `no_less_exact` allows for measuring it."""
    M, K, N, dtype, layout = shape
    config = config or tune.reference(*shape)
    x1, x2 = tune.operands(M, K, N, dtype, layout, torch.Generator(device="cuda").manual_seed(9))
    ref = torch.mm(x1.double().contiguous(), x2.double().contiguous())
    err = lambda c: ((ext.matrix_mul(x1, x2, c) - ref).norm() / ref.norm()).item()
    now, before = err(None), err(config)
    print(shape, tune.pick(*shape), now, config, before, flush=True)
    assert now <= before * tune.ERROR_SLACK ** 0.5 + 1e-10
