"""The single track's norms and the products behind them, one kernel each (single_step.hip)."""

import pytest
import torch


def _block(pkg, heads, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        blk = pkg.nn.PairformerBlock(n_heads=heads)
    with torch.no_grad():
        for name, p in blk.named_parameters():
            p.normal_(0.0, 0.05, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    blk.invalidate()
    return blk


# one row; one short of a tile of 32 and one past it; the last size of the kernels and the first behind it; heads of 24, 32 and 48
@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,heads", [(1, 16), (31, 16), (33, 16), (64, 12), (161, 8), (400, 16), (401, 16)])
def test_single_update_is_as_exact_as_with_two_kernels_each(gpu_pkg, n, heads, io):
    """Rounded at the same places; only fp32 sums have another order, 1e-6 of a value, so that few roundings to bf16 fall on the other
    side.  Against the fp32 check mode the error is therefore that of the separate kernels (a hook makes the block run module by
    module): by root mean square up to a flip of some values in a hundred, 5 %; the largest of up to 150000 by one flip more, a half."""
    blk = _block(gpu_pkg, heads, n)
    gen = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(io)
    pair, single, seq = rnd(n, n, 128), rnd(n, 384) * 2 + 3, (torch.arange(n, device="cuda") < n - n // 10).float()
    mask = (seq[:, None] * seq[None, :]).contiguous()
    got = blk(pair.clone(), mask, single.clone(), seq)[1]
    hook = blk.single_attention_.adaptive_layernorm.register_forward_hook(lambda m, args, out: None)
    apart = blk(pair.clone(), mask, single.clone(), seq)[1]
    hook.remove()
    with gpu_pkg.nn.check_mode():
        want = blk(pair.float(), mask, single.float(), seq)[1].double()
    assert got.dtype == io and torch.isfinite(got).all()
    error, allowed = (got.double() - want).abs(), (apart.double() - want).abs()
    update = (want - single.double()).square().mean().sqrt()
    assert 0 < allowed.square().mean().sqrt() <= 1e-2 * (want.square().mean().sqrt() if io == torch.bfloat16 else update)
    assert error.square().mean().sqrt() <= 1.05 * allowed.square().mean().sqrt() and error.max() <= 1.5 * allowed.max()
