"""Row splits of column sums (csrc/reduce.hip, reduce_geom), seen through the
workspace a sum asks for: splits x slabs of columns x 1 KiB."""

import pytest

from tilec import _lib


@pytest.mark.parametrize("R,splits", [(256, 1), (511, 1), (512, 4), (1024, 8), (4096, 32), (5000, 32), (8192, 32),
                                      (10000, 37), (65536, 256), (1 << 20, 512)])
def test_splits_of_a_narrow_matrix(R, splits):
    """One slab of columns: 2 blocks a wave up to 32 splits, 4 beyond, at most
    512; rows per split are whole blocks of 16."""
    need = _lib.lib().tilec_sum_workspace_bytes(R, 8, 0, _lib.F32, 0)
    assert need == (splits * 1024 if splits > 1 else 0), need / 1024
