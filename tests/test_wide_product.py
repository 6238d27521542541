"""Products of K = 384 with very many fp32 results (wide_product.hip): the bits of the general kernel."""

import pytest
import torch


# the first size of the kernel, and a strip of columns less; one row more than whole panels, one less; parts of one panel's rest; the
# fewest columns; rows and columns of wider matrices
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,bias,sigmoid", [(200, 73472, True, False), (200, 73344, True, False), (193, 98304, False, True),
                                              (255, 61440, True, True), (769, 36864, True, False), (4865, 3072, False, False)])
def test_as_in_pieces(gpu_pkg, m, n, bias, sigmoid):
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, 384, generator=g, device="cuda").bfloat16()
    w = torch.randn(n, 384, generator=g, device="cuda").bfloat16()
    b = torch.randn(n, generator=g, device="cuda") if bias else None
    out = torch.full((m + 1, n), 7.0, device="cuda")
    got = gpu_pkg.ops.linear(x, w, bias=b, out_dtype=torch.float32, sigmoid=sigmoid, alpha=0.5, out=out[:m])
    step = 1536                                   # (too few columns for the kernel)
    for c in range(0, n, step):
        e = min(c + step, n)
        part = gpu_pkg.ops.linear(x, w[c:e], bias=None if b is None else b[c:e], out_dtype=torch.float32, sigmoid=sigmoid, alpha=0.5)
        assert torch.equal(got[:, c:e], part)
    assert (out[m] == 7.0).all()
