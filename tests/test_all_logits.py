"""The pair logits of all super-blocks of a token transformer in one launch: the bits of one launch each."""

import pytest
import torch


# a pixel; a quad with a rest; queries past a tile of 32; rows of heads past 32, a block of them cut short
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 5, 33, 100])
@pytest.mark.parametrize("heads", [64, 104, 384])
@pytest.mark.parametrize("quads", [True, False])
def test_as_64_heads_at_a_time(gpu_pkg, n, heads, quads):
    g = torch.Generator(device="cuda").manual_seed(n + heads)
    pair, ln = torch.randn(n, n, 128, generator=g, device="cuda"), torch.rand(128, generator=g, device="cuda")
    w = torch.zeros((heads + 31) // 32 * 32, 128, device="cuda").bfloat16()
    w[:heads] = torch.randn(heads, 128, generator=g, device="cuda")
    got = gpu_pkg.ops.pair_logits(pair, ln, None, w, heads, quads=quads)
    for h in range(0, heads, 64):
        k = min(64, heads - h)
        assert torch.equal(got[h:h + k], gpu_pkg.ops.pair_logits(pair, ln, None, w[h:h + 64].contiguous(), k, quads=quads))


# super-blocks together, one alone, and projections that no whole blocks of 32 rows make
@pytest.mark.gpu
@pytest.mark.parametrize("blocks,size", [(6, 2), (4, 4), (3, 1)])
@pytest.mark.parametrize("n", [24, 21])
def test_super_blocks(gpu_pkg, blocks, size, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionTransformer(num_blocks=blocks, super_block_size=size)
    pair = torch.randn(n, n, 128, generator=g, device="cuda")
    got = mod.pair_logits(pair)
    assert len(got) == blocks // size
    for m, l in zip(mod.pair_logits_projection, got):
        w = gpu_pkg.nn.base.pad_rows(m.weight.detach().bfloat16(), 32)
        want = gpu_pkg.ops.pair_logits(pair, mod.packed()["ln_w"], None, w, size * 16, quads=n % 4 == 0)
        assert torch.equal(l.reshape(want.shape), want)
