"""The pair operators at the sizes where a tile's steps go to four, two or one
workgroup (the prologue of the triangle multiplication) and to three or one (the
projections of the triangle attention), with whole tiles of masked positions at
the end, at both widths; against the float64 CPU oracle."""

import pytest
import torch

from oracle import af3_oracle as O

pytestmark = pytest.mark.gpu
D = torch.float64


@pytest.mark.parametrize("c", [128, 64])
@pytest.mark.parametrize("n", [152, 160, 181, 219, 224])
def test_steps_dealt_to_workgroups(gpu_pkg, n, c):
    g = torch.Generator().manual_seed(n)
    pair = O.round_bf16(torch.randn(n, n, c, generator=g))
    mask = (torch.rand(n, n, generator=g) > 0.2).float()
    mask[:, 0] = 1
    mask[n - 3:] = 0
    p = {k: O.round_bf16(v) for k, v in O.make_triangle_multiplication_params(g, c, std=0.1).items()}
    q = {k: O.round_bf16(v) for k, v in O.make_grid_self_attention_params(g, c, 4, std=0.1).items()}
    tri = gpu_pkg.nn.TriangleMultiplication(c_pair=c, _outgoing=True)
    att = gpu_pkg.nn.GridSelfAttention(c_pair=c, num_head=4, transpose=True)
    for mod, params, want in (
            (tri, p, O.triangle_multiplication(pair.to(D), mask.to(D), O.cast_params(p, D), True)),
            (att, q, O.grid_self_attention(pair.to(D), mask.to(D), O.cast_params(q, D), 4, True))):
        mod.load_state_dict(params)
        mod.to("cuda:0")
        got = mod(pair.to("cuda:0"), mask.to("cuda:0")).cpu().to(D)
        scale = float((want ** 2).mean().sqrt())
        rms, mx = float(((got - want) ** 2).mean().sqrt()) / scale, float((got - want).abs().max()) / scale
        assert torch.isfinite(got).all() and rms <= 1e-2 and mx <= 8e-2, (type(mod).__name__, rms, mx)
