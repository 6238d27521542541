"""The adaptive norm of 768 channels (ln_rows_768_kernel): twelve channels to a lane, several rows of a token to a wave."""

import pytest
import torch


# one sample; as many as a wave takes and one more, shared out evenly; one token, and tokens that leave waves of a workgroup without one
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("samples,tokens", [(1, 1), (1, 67), (2, 5), (3, 33), (4, 13), (5, 6), (6, 9), (7, 1), (11, 21)])
def test_rows_of_a_token_together(gpu_pkg, samples, tokens, dtype):
    g = torch.Generator(device="cuda").manual_seed(100 * samples + tokens)
    x = (torch.randn(samples * tokens, 768, generator=g, device="cuda") * 3 + 1).to(dtype)
    ss = torch.randn(tokens, 4 * 768, generator=g, device="cuda")
    scale, shift = ss[:, 768:1536], ss[:, 1536:2304]
    y = gpu_pkg.ops.layer_norm(x, scale=scale, shift=shift)
    n = torch.nn.functional.layer_norm(x.double(), (768,))
    want = torch.sigmoid(scale.double()).repeat(samples, 1) * n + shift.double().repeat(samples, 1)
    assert ((y.double() - want).abs() <= 1.01 * 2.0 ** -8 * want.abs() + 1e-4).all()
    # a row's result is its own: the same bits with every row's conditioning written out
    assert torch.equal(y, gpu_pkg.ops.layer_norm(x, scale=scale.repeat(samples, 1), shift=shift.repeat(samples, 1)))


# 1e22 squared is past fp32: the variance is an infinity, 1 / sqrt of it zero, and the row its shift; an infinity or NaN in a row is a
# NaN in all of it and nowhere else
@pytest.mark.gpu
@pytest.mark.parametrize("samples", [1, 5])
def test_infinities(gpu_pkg, samples):
    g = torch.Generator(device="cuda").manual_seed(samples)
    x = torch.randn(samples * 6, 768, generator=g, device="cuda").bfloat16()
    ss = torch.randn(6, 2 * 768, generator=g, device="cuda")
    clean = gpu_pkg.ops.layer_norm(x, scale=ss[:, :768], shift=ss[:, 768:])
    y = x.clone()
    y[0] *= 1e22
    y[1, 767], y[2, 3], y[3, 600] = float("inf"), float("nan"), float("-inf")
    got = gpu_pkg.ops.layer_norm(y, scale=ss[:, :768], shift=ss[:, 768:])
    assert torch.equal(got[0], ss[0, 768:].bfloat16())
    assert got[1:4].isnan().all() and torch.equal(got[4:], clean[4:])
