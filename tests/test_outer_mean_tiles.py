"""The outer-product mean's three tile heights (contract.hip) against the fp32 check mode."""

import pytest
import torch


# tokens x MSA rows on either side of the lines between the heights; ragged in both; one token; K past one slab
@pytest.mark.gpu
@pytest.mark.parametrize("n,rows", [(1, 3), (7, 8), (33, 70), (64, 600), (65, 600), (90, 512), (97, 512), (161, 66), (187, 301),
                                    (193, 1024), (300, 1024), (301, 40)])
def test_every_tile_height_against_fp32(gpu_pkg, n, rows):
    g = torch.Generator(device="cuda").manual_seed(n)
    mod = gpu_pkg.nn.OuterProductMean().to("cuda")
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.1, generator=g)
    mod.invalidate()
    msa = torch.randn(rows, n, 64, generator=g, device="cuda").bfloat16().float()
    mask = (torch.rand(rows, n, generator=g, device="cuda") > 0.1).float()
    mask[0] = 1.0
    got = mod(msa, mask)
    with gpu_pkg.nn.check_mode(True):
        want = mod(msa, mask)
    scale = want.square().mean().sqrt()
    # bf16 operands and bf16 outer products in between: the bound of every bf16 operator against this mode
    assert torch.isfinite(got).all() and (got - want).square().mean().sqrt() <= 1e-2 * scale and (got - want).abs().max() <= 8e-2 * scale
