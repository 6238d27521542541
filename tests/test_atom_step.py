"""The tail of an atom transformer block in one kernel (atom_step.hip) against the operators one by one."""

import pytest
import torch


# atoms that fill no tile of 32 and that do; one sample and several; fewer tiles than XCDs; transitions of one to eight
# blocks of 32 hidden units (a factor of 3 has no such kernel)
@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("samples,s,q,k,factor", [(1, 1, 1, 4, 2), (2, 3, 7, 12, 1), (3, 2, 32, 16, 2), (1, 9, 32, 128, 2), (5, 13, 31, 60, 2)])
def test_the_steps_give_the_bits_of_the_operators(gpu_pkg, samples, s, q, k, factor, io):
    g = torch.Generator(device="cuda").manual_seed(s * q)
    rnd = lambda *d: torch.randn(*d, generator=g, device="cuda")
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionCrossAttTransformer()
        for tr in mod.transition_block:
            tr.__init__(c_x=128, c_single_cond=128, num_intermediate_factor=factor, use_single_cond=True)
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.08, generator=g)
    mod.invalidate()
    idx = torch.randint(0, s * q, (s, k), generator=g, device="cuda")
    gather = (idx, torch.rand(s, k, generator=g, device="cuda") > 0.2)
    act, mk = rnd(samples, s, q, 128).to(io), gather[1].float()
    mq = (torch.rand(s, q, generator=g, device="cuda") > 0.2).float()
    sq = rnd(s, q, 128)
    sk = sq.view(s * q, 128)[idx] * gather[1][..., None]
    cond = mod.conditioning(sq, sk, rnd(s, q, k, 16), keys_are_query_atoms=gather)
    run = lambda: mod(act.clone(), mq, gather, mk, sq, sk, None, cond=cond)
    want, seen = run(), []
    hook = mod.transition_block[1].adaptive_layernorm.register_forward_hook(lambda *a: seen.append(1))
    got = run()
    hook.remove()
    assert seen and want.dtype == io and torch.isfinite(want).all() and not torch.equal(want, act) and torch.equal(got, want)
