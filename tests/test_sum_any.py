"""Sums of rows that are not whole 16-byte groups (csrc/reduce.hip, kAny): the
moved last group counts every element once and no load leaves its row, over
lengths around a group, a lane's groups and a split; then the kernels
themselves against the fp64 oracle, with NaN in every element outside x."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tilec import ext


def row_geom(R, C, E):
    """reduce_geom of row sums: lanes per row, columns per split."""
    cd = lambda a, b: -(-a // b)
    lpr = 1
    while lpr < min(64, max(1, cd(C, 4 * E))):
        lpr *= 2
    cells = cd(max(R, 1), 4 * (64 // lpr))
    s = max(1, min(cd(512, cells), C // (64 * E * 8))) if lpr == 64 and cells < 512 else 1
    return lpr, max(64 * E, cd(cd(C, s), 64 * E) * 64 * E)


@pytest.mark.parametrize("E", [4, 8])
def test_row_groups_cover_each_element_once(E):
    for R, C in [(300, c) for c in (E, E + 1, 4 * E, 4 * E + 1, 65, 129, 64 * 4 * E - 1, 64 * 4 * E + 1)] + [
            (3, 64 * E * 16 + 1), (3, 64 * E * 17 - 1), (2, 64 * E * 48 + E - 1), (1, 200003)]:
        lpr, chunk = row_geom(R, C, E)
        U, step = 16 if lpr == 64 else 4, E * lpr
        seen = np.zeros(C, int)
        for cbeg in range(0, C, chunk):
            cols = min(C, cbeg + chunk) - cbeg
            back = min(cbeg, E)
            groups = np.arange(0, -(-cols // (U * step)) * U * step, E)
            b = groups // (U * step) * U * step
            full = b + U * step <= cols
            loaded = full | (groups // step * step < cols)
            at = np.where(full, groups, np.minimum(groups, cols - E))[loaded]
            drop = np.where(full, 0, groups - (cols - E))[loaded]
            assert (at + back).min() >= 0 and (at + cbeg).min() >= 0 and (at + cbeg + E).max() <= C
            for e in range(E):
                np.add.at(seen, (at + cbeg + e)[e >= drop], 1)
        assert (seen == 1).all(), (R, C)


@pytest.mark.parametrize("E", [4, 8])
def test_column_groups_land_on_their_columns(E):
    for C in (E, E + 1, 2 * E - 1, 16 * E - 1, 16 * E + 1, 17 * E - 1, 17 * E + 1, 33 * E - 2):
        got = np.full(C, -1)
        for n0 in range(0, C, 16 * E):
            back = min(n0, E)
            for q in range(16):
                cn = C - (n0 + E * q)
                col = min(E * q, C - E - n0) + back
                first = n0 - back + col
                assert col >= 0 and 0 <= first and first + E <= C
                acc = list(range(first, first + E))  # which column each accumulator sums
                i = cn
                while 0 < i < E:
                    acc = acc[1:] + [-1]
                    i += 1
                for e in range(E):
                    if n0 + E * q + e < C:
                        got[n0 + E * q + e] = acc[e]
        assert (got == np.arange(C)).all(), C


SHAPES = [(1, 9), (5, 8), (300, 17), (70, 33), (129, 257), (16, 1025), (17, 2049), (3, 100003), (4097, 129),
          (100001, 9), (1000, 4097),
          (511, 65), (512, 65), (640, 24)]  # column sums split from 512 rows on


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("gap,shift", [(0, 0), (0, 1), (3, 1), (8, 3)])
def test_any_alignment(dtype, gap, shift):
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    for i, (R, C) in enumerate(SHAPES):
        x = O.normal((R, C), 1600 + i)
        if dtype == "bf16":
            x = O.bf16_to_f32(O.bf16_round(x))
        flat = torch.full((shift + R * (C + gap) + 16,), float("nan"), dtype=dt, device="cuda")
        v = flat.as_strided((R, C), (C + gap, 1), shift)
        v.copy_(torch.from_numpy(x).to("cuda").to(dt))
        for axis in (0, 1):
            print("sum", dtype, "axis", axis, (R, C), "gap", gap, "shift", shift, flush=True)
            got = ext.sum(v, axis)
            torch.cuda.synchronize()
            assert O.sum_error_ok(got.cpu().numpy(), x, axis), (R, C, axis)
