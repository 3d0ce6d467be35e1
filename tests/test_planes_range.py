"""Values far apart in one product on the fp32 plane kernels
(csrc/gemm_f32_x6.hip): every element's split is exact by itself, whatever
else its row or column holds."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import _lib, ext

PLANES = [v["name"] for v in _lib.variants() if v["name"].endswith("_x6")]


def bf16(x):
    return O.bf16_to_f32(O.bf16_round(x))


def test_split_is_exact_for_every_exponent():
    """The kernel's split in numpy: hi + mid + lo == 2^16 x for magnitudes from
    fp32's smallest subnormal to 2^111, and its planes are finite."""
    rng = np.random.default_rng(5)
    for e in range(-149, 111):
        x = np.ldexp(rng.uniform(1, 2, 256), e).astype(np.float32) * rng.choice([-1, 1], 256).astype(np.float32)
        rest = y = x * np.float32(2**16)
        planes = []
        for _ in range(3):
            planes.append(bf16(rest))
            rest = (rest - planes[-1]).astype(np.float32)
        assert np.isfinite(planes).all() and (np.sum(planes, axis=0, dtype=np.float64) == y.astype(np.float64)).all(), e


# A product of one term: the three dropped plane products are at most 2 x 2^-9 x 2^-17 of it, and at most six
# roundings of 2^-24 follow
ONE = 8 * 2.0**-24


@pytest.mark.gpu
@pytest.mark.parametrize("name", PLANES)
def test_one_term_beside_large_values(name):
    """x2's columns pick one element of each x1 row, of magnitude 2^e, beside
    ordinary ones; the other way round too."""
    es = np.arange(-126, 111)
    k, n = 48, 80
    a, sel = O.normal((len(es), k), 3), np.zeros((k, n), np.float32)
    c = (1 + np.abs(O.normal((len(es),), 4)) % 1).astype(np.float32)
    a[:, 20] = np.ldexp(c, es).astype(np.float32)
    for s in (0, 40, -40):  # the picking value; results that are normal numbers
        sel[20, :] = np.float32(2.0**s * 1.2345)
        ok = (es + s >= -126) & (es + s < 127)
        for x1, x2, t in ((a, sel, False), (np.ascontiguousarray(sel.T), np.ascontiguousarray(a.T), True)):
            got = ext.matrix_mul(torch.from_numpy(x1).cuda(), torch.from_numpy(x2).cuda(), (name, 1)).cpu().numpy()
            want = x1.astype(np.float64) @ x2.astype(np.float64)
            got, want = (got.T, want.T) if t else (got, want)
            err = (np.abs(got - want) / np.abs(want))[ok].max()
            print(name, "picked by 2^%d" % s, "x2 holds them" if t else "x1 holds them", err, flush=True)
            assert err <= ONE


@pytest.mark.gpu
@pytest.mark.parametrize("name", PLANES)
def test_scales_along_k(name):
    """(x1 D)(D^-1 x2) with D alternating between d and 1 / d: every factor is a
    normal fp32 number and so is every product."""
    m, k, n = 130, 256, 140
    a, b = O.normal((m, k), 5), O.normal((k, n), 6)
    for d in (1e30, 1e33, 1e36, 1e37):
        s = np.where(np.arange(k) % 2, d, 1 / d)
        x1, x2 = (a * s).astype(np.float32), (b / s[:, None]).astype(np.float32)
        got = ext.matrix_mul(torch.from_numpy(x1).cuda(), torch.from_numpy(x2).cuda(), (name, 1)).cpu().numpy()
        err = O.rel_l2(got, O.matmul_f64(x1, x2))
        print(name, d, err, flush=True)
        # 6 K / 16 = 96 roundings of the sum, or 256 on the fp32 MFMAs: sqrt(256) 2^-25, and twice that
        assert err <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("name", PLANES)
def test_subnormals(name):
    """A subnormal against a value that lifts it back: 2^-140 x 2^126."""
    x1, x2 = np.ones((70, 33), np.float32), np.zeros((33, 66), np.float32)
    x1[:, 7] = np.ldexp(1.0, -140)
    x2[7, :] = np.ldexp(1.0, 126)
    for a, b in ((x1, x2), (np.ascontiguousarray(x2.T), np.ascontiguousarray(x1.T))):
        got = ext.matrix_mul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), (name, 1))
        assert (got == 2.0**-14).all()
