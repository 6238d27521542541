"""The triangle contraction on either side of the line between its two kernels."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("n", [127, 129, 160, 187, 192, 193, 200])
def test_contraction_around_the_line(gpu_pkg, n):
    """T[c] = A[c] B[c]^T: fp32 sums of bf16 products, one rounding to bf16 (half a unit in 2^8, and the sums' order)."""
    g = torch.Generator(device="cuda").manual_seed(n)
    np_ = (n + 7) // 8 * 8
    a, b = (torch.zeros(128, n, np_, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    for x in (a, b):
        x[..., :n] = torch.randn(128, n, n, generator=g, device="cuda")
    got = gpu_pkg.ops.triangle_contraction(a, b)[..., :n].double()
    want = torch.bmm(a[..., :n].double(), b[..., :n].double().transpose(1, 2).contiguous())
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * n ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,n,k", [(8, 129, 1024, 136), (8, 160, 2400, 160), (8, 200, 3328, 200), (8, 200, 3080, 200), (3, 300, 9000, 304)])
def test_batched_products_around_the_line(gpu_pkg, batch, m, n, k):
    """Up to a hundred large tiles on the general kernel, more on the large tile (104, 96, 108)."""
    g = torch.Generator(device="cuda").manual_seed(m)
    a, b = (torch.randn(batch, r, k, generator=g, device="cuda").bfloat16() for r in (m, n))
    got = torch.empty(batch, m, n, device="cuda", dtype=torch.bfloat16)
    lib = gpu_pkg.lib.load()
    rc = lib.af3_batched_nt_product_forward(a.data_ptr(), b.data_ptr(), got.data_ptr(), batch, m, n, k,
                                            torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = torch.bmm(a.double(), b.double().transpose(1, 2).contiguous())
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * k ** 0.5).all()
