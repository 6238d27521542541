"""Heads of 48 over plain keys (attention.hip, token_attention_kernel) against the general form of the same arithmetic."""

import pytest
import torch


# keys that fill no tile of 64, one, two and three of them, and a few past a tile; queries of one and of two tiles of 128; the mask
# over the end of a sequence, its first tile, single keys and a whole sequence
@pytest.mark.gpu
@pytest.mark.parametrize("batch,n,mask", [(1, 4, "end"), (3, 36, "some"), (2, 64, "none"), (5, 68, "end"), (2, 124, "first"), (1, 128, "all"),
                                          (2, 132, "some"), (1, 192, "first"), (5, 200, "end"), (2, 324, "some"), (1, 516, "first")])
def test_token_attention_gives_the_bits_of_the_general_form(gpu_pkg, batch, n, mask):
    """A bias that does not begin on 16 bytes takes the general form; both orders of an aligned one take the kernel."""
    g = torch.Generator(device="cuda").manual_seed(batch * n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, h = 768, 16
    x, w, qb = rnd(batch, n, c).bfloat16(), (rnd(4 * c, c) * 0.05).bfloat16(), rnd(c)
    logits = rnd(h, n, n) * 3
    logits[:, 0] += 40                                       # a row whose maximum moves the base
    logits[:, -1] *= 10
    keep = torch.ones(n, device="cuda")
    if mask == "end":
        keep[n - n // 8 - 1:] = 0
    elif mask == "first":
        keep[:70] = 0
    elif mask == "some":
        keep[::3] = 0
    elif mask == "all":
        keep[:] = 0
    off = torch.empty(logits.numel() + 1, device="cuda")[1:].view_as(logits)
    off.copy_(logits)
    run = lambda b: gpu_pkg.ops.batch_diffusion_self_attention(x, keep, b, w, qb, h, out_dtype=torch.float32)
    want = run(off)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    assert torch.equal(run(logits), want) and torch.equal(run(gpu_pkg.ops.quad_major_bias(logits)), want)
    one = gpu_pkg.ops.batch_diffusion_self_attention(x[:1].contiguous(), keep, logits, w, qb, h, out_dtype=torch.float32)
    assert torch.equal(one, run(logits).view(batch, n, c)[:1].reshape(one.shape))
