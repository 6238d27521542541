"""Triangle attention core: where a row's first live key tile is not the one a workgroup asks for first."""

import pytest
import torch

from test_gpu_parity import dev, gen, rb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,first", [(33, 5), (70, 64), (200, 64), (200, 130), (330, 64), (330, 193), (1100, 1025)])
def test_rows_that_begin_with_masked_keys(gpu_pkg, n, first):
    """Keys below `first` are masked in every row but some (whole tiles of them from 64 on); 330 and 1100 tokens take two rows
    to a wave, 1100 more than one batch of mask values.  Bounds as in test_kernel_level_attention_core."""
    g, d = gen(n + first), dev()
    q, k, v = (rb(torch.randn(n, 4, n, 32, generator=g) * 0.7).to(d) for _ in range(3))
    bias = rb(torch.randn(4, n, n, generator=g)).half().float().to(d)
    mask = torch.ones(n, n)
    mask[:, :first] = 0
    mask[4::7] = 1                       # these rows live from the first key on
    mask[5::7, first + 1:] = 0           # these have one live key
    mask[6::7] = 0                       # these have none
    mask = mask.to(d)
    run = lambda m: gpu_pkg.ops.grid_attention_core(q.bfloat16(), k.bfloat16(), gpu_pkg.ops.pack_vt(v.transpose(-1, -2).bfloat16()),
                                                    gpu_pkg.ops.pack_pair_bias(bias), m)
    og = run(mask).view(n, n, 4, 32).double()
    err = ref = worst = 0.0
    for b in range(0, n, 64):
        logits = (q[b:b + 64].double() @ k[b:b + 64].double().transpose(-1, -2) + bias.double()) / 1.4426950408889634
        logits = logits.masked_fill(mask[b:b + 64, None, None, :] == 0, -1e9)
        want = (torch.softmax(logits, -1) @ v[b:b + 64].double()).permute(0, 2, 1, 3)
        diff = og[b:b + 64] - want
        err, ref, worst = err + diff.square().sum().item(), ref + want.square().sum().item(), max(worst, diff.abs().max().item())
    rms = (ref / og.numel()) ** 0.5
    assert (err / ref) ** 0.5 < 5e-3 and worst / rms < 7e-2
    assert torch.equal(run(None), run(torch.ones_like(mask)))
