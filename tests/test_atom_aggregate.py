"""Atoms to tokens in one kernel (atom_aggregate.hip)."""

import pytest
import torch


# tokens beside a multiple of four; one octet of slots to four, with a rest; tokens without an atom; more units than workgroups
@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,slots", [(1, 1, 24), (5, 4, 24), (2, 7, 1), (3, 66, 8), (1, 5, 13), (4, 33, 32), (5, 411, 24)])
def test_as_product_and_gather(gpu_pkg, batch, tokens, slots):
    """The same products rounded to the same bf16, up to 32 of them summed in another order: 32 rounding errors of the sum."""
    g = torch.Generator(device="cuda").manual_seed(tokens * slots)
    n_src = tokens * slots + 5
    x = torch.randn(batch, n_src, 128, generator=g, device="cuda").bfloat16()
    w = (torch.randn(768, 128, generator=g, device="cuda") * 0.1).bfloat16()
    idx = torch.randint(0, n_src, (tokens, slots), generator=g, device="cuda").int()
    live = torch.randint(0, slots + 1, (tokens, 1), generator=g, device="cuda")      # a token's first slots, but for some
    idx[(torch.arange(slots, device="cuda") >= live) | (torch.rand(tokens, slots, generator=g, device="cuda") < 0.1)] = -1
    dead = torch.ones(n_src, dtype=torch.bool, device="cuda")
    dead[idx[idx >= 0].long()] = False
    x[:, dead] = float("nan")                                                        # (read by nobody)
    count = (idx >= 0).sum(-1).float().clamp(min=1e-10)
    frags = gpu_pkg.nn.base.fragments(w).reshape(768, 128)
    got = gpu_pkg.ops.atom_aggregate(x, idx, count, frags)
    want = gpu_pkg.ops.gathered_relu_mean(gpu_pkg.ops.linear(x, w), idx, count)
    assert (got - want).abs().max() <= 32 * 2.0 ** -24 * want.max() * slots
    assert (got[:, (idx < 0).all(-1)] == 0).all()


def test_refused(pkg):
    lib = pkg.lib.load()
    one = 1 << 20
    assert lib.af3_atom_aggregate_forward(one, None, one, one, one, 1, 8, 8, 4, None) == -1
    assert lib.af3_atom_aggregate_forward(one, one, one, one, one, 1, 8, 8, 33, None) == -1
    assert lib.af3_atom_aggregate_forward(one + 2, one, one, one, one, 1, 8, 8, 4, None) == -1
