"""fp32 products over one k are correctly rounded, whatever the library's own
rule runs (the plane kernels' dropped terms would show there)."""

import pytest
import torch

from tilec import _lib, ext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(65, 63), (2000, 3000), (2049, 2048), (4096, 4096)])
def test_one_product_is_correctly_rounded(m, n):
    g = torch.Generator(device="cuda").manual_seed(m)
    a, b = torch.randn(m, 1, generator=g, device="cuda"), torch.randn(1, n, generator=g, device="cuda")
    for layout in range(4):
        x1 = a.t().contiguous().t() if layout & 1 else a
        x2 = b.t().contiguous().t() if layout & 2 else b
        assert torch.equal(ext.matrix_mul(x1, x2, (_lib.VARIANT_AUTO, 0)), a * b), layout
