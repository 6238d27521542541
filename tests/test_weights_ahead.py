"""The token transformer's norms have workgroups that read what the kernels behind them will (rowops.hip, weights and pair
logits): nothing of it shows in the results."""

import pytest
import torch


# channels: just past the narrow norm, 3 and 4 chunks of 512; rows: fewer than one workgroup, ragged; logits past 4 MB
@pytest.mark.gpu
@pytest.mark.parametrize("c,heads,samples,n", [(144, 3, 1, 3), (384, 8, 2, 21), (1056, 22, 1, 30), (1536, 32, 3, 9), (768, 16, 1, 300)])
def test_one_call_gives_the_bits_of_its_operators(gpu_pkg, c, heads, samples, n):
    g = torch.Generator(device="cuda").manual_seed(c + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionTransformer(c_act=c, num_head=heads, num_blocks=2, super_block_size=1)
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.05, generator=g)
    mod.invalidate()
    act, cond, pair = rnd(samples, n, c).bfloat16(), rnd(n, 384), rnd(n, n, 128)
    mask = (torch.arange(n, device="cuda") < n - 1).float()
    run = lambda: mod(act.clone(), mask, cond, pair)
    want, seen = run(), []
    hook = mod.self_attention[1].adaptive_layernorm.register_forward_hook(lambda *a: seen.append(1))
    got = run()
    hook.remove()
    assert seen and torch.isfinite(want).all() and torch.equal(got, want)
