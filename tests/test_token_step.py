"""The token transformer's kernels (token_step.hip) against the operators one by one."""

import ctypes

import pytest
import torch

from bf16_tolerances import RMS_TOL, cap
from oracle import af3_oracle as O


# tiles hold all samples of 4 to 16 tokens, by the number of samples and of tiles: one token, tiles that are filled and that are
# not, both sizes of every number of samples, one number that has no such kernel, more tokens than it takes, weights of 6 to 18 tiles;
# products over rows: a row and two past a tile of 64, the most that the gated product of few rows takes and one more, the most for
# all three and one tile more
@pytest.mark.gpu
@pytest.mark.parametrize("samples,n,factor", [(1, 1, 2), (1, 33, 2), (1, 64, 1), (1, 200, 2), (1, 337, 2), (2, 17, 2), (2, 161, 1), (3, 31, 2),
                                              (3, 155, 2), (4, 40, 3), (4, 81, 2), (5, 6, 2), (5, 77, 2), (5, 100, 2), (5, 130, 2), (6, 11, 2),
                                              (6, 21, 2), (6, 112, 1), (6, 113, 2), (7, 384, 2), (7, 385, 2)])
def test_the_steps_give_the_bits_of_the_operators(gpu_pkg, samples, n, factor):
    g = torch.Generator(device="cuda").manual_seed(100 * samples + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionTransformer(num_blocks=2, super_block_size=1)
        for tr in mod.transition_block:
            tr.__init__(c_x=768, c_single_cond=384, num_intermediate_factor=factor, use_single_cond=True)
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.05, generator=g)
    mod.invalidate()
    act, cond, pair = rnd(samples, n, 768).bfloat16(), rnd(n, 384), rnd(n, n, 128)
    act[0, 0] *= 1000                                            # rows of other sizes
    act[-1, -1] = 0
    mask = (torch.arange(n, device="cuda") < max(1, n - 1)).float()
    run = lambda: mod(act.clone(), mask, cond, pair)
    want, seen = run(), []
    hook = mod.self_attention[1].adaptive_layernorm.register_forward_hook(lambda *a: seen.append(1))
    got = run()
    hook.remove()
    assert seen and torch.isfinite(want).all() and not torch.equal(want, act) and torch.equal(got, want)


# tiles of 96 and of 128 rows in every product, the last one short, full and by a row too long; hidden layers of 768 and 1536
@pytest.mark.gpu
@pytest.mark.parametrize("samples,n,factor", [(7, 95, 2), (6, 112, 1), (7, 137, 2), (7, 141, 1), (6, 160, 2), (7, 391, 2), (7, 384, 1), (6, 641, 2),
                                              (7, 577, 1)])
def test_rows_in_larger_tiles(gpu_pkg, samples, n, factor):
    test_the_steps_give_the_bits_of_the_operators(gpu_pkg, samples, n, factor)


@pytest.mark.gpu
@pytest.mark.parametrize("samples,n", [(1, 40), (5, 100), (6, 20)])
def test_a_null_plane_of_logits_is_no_bias(gpu_pkg, samples, n):
    """The library call takes one pointer to pair logits for each block; the bits of logits that are zero."""
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionTransformer(num_blocks=2, super_block_size=1)
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.05, generator=g)
    lib, L, c = gpu_pkg.lib.load(), gpu_pkg.lib, 768
    table = gpu_pkg.nn.diffusion_transformer.block_table(mod, mod._blocks(), c)
    act, ss, gate = rnd(samples, n, c).bfloat16(), rnd(n, 4, 2 * c), torch.sigmoid(rnd(n, 4, c))
    logits, zeros, outs = rnd(16, n, n), torch.zeros(16, n, n, device="cuda"), []
    need = lib.af3_diffusion_transformer_workspace_bytes(samples, n, c, table.hidden)
    for second in (zeros.data_ptr(), None):
        x, ws = act.clone(), torch.empty(need, dtype=torch.uint8, device="cuda")
        planes = (ctypes.c_void_p * 2)(logits.data_ptr(), second)
        L.check(lib.af3_diffusion_transformer_forward(
            table, 2, x.data_ptr(), L.AF3_BF16, samples, n, c, table.hidden, 16, None, planes, 0, ss.data_ptr(), gate.data_ptr(), n,
            ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream), "transformer")
        outs.append(x)
    assert torch.isfinite(outs[0]).all() and not torch.equal(outs[0], act) and torch.equal(*outs)


# norm and product in one kernel with the gated one (one to five samples, the most rows of either, one more), in kernels of their own
# (2688 rows are the most for all three products, 2695 take one of them)
@pytest.mark.gpu
@pytest.mark.parametrize("samples,n", [(1, 33), (3, 100), (5, 126), (5, 134), (5, 135), (7, 384), (7, 385)])
def test_a_bf16_stream_against_the_oracle(gpu_pkg, samples, n):
    """The update of two blocks to the tolerances of an fp32 stream, and four roundings of the stream to 8 bits on top: each at most
    2^-9 of a value, of their rms no more than that (independent: twice for four) and at most four times at any place."""
    g = torch.Generator().manual_seed(n)
    rb = O.round_bf16
    p = {k: rb(v) for k, v in O.make_diffusion_transformer_params(g, num_blocks=2, super_block_size=2, std=0.05).items()}
    mod = gpu_pkg.nn.DiffusionTransformer(num_blocks=2, super_block_size=2)
    mod.load_state_dict(p)
    mod = mod.cuda()
    act, cond, pair = (rb(torch.randn(*s, generator=g)).cuda() for s in ((samples, n, 768), (n, 384), (n, n, 128)))
    mask = (torch.arange(n, device="cuda") < n - n // 8).float()
    got = mod(act.bfloat16(), mask, cond, pair).double()
    want = O.diffusion_transformer(act.double(), mask.double(), cond.double(), pair.double(), {k: v.double().cuda() for k, v in p.items()}, 16, 2, 2)
    rms = lambda x: x.pow(2).mean().sqrt()
    scale = rms(want - act)
    assert rms(got - want) <= RMS_TOL * scale + 2 * 2.0 ** -9 * rms(want)
    assert (got - want).abs().max() <= cap("diffusion_transformer") * scale + 4 * 2.0 ** -9 * want.abs().max()
