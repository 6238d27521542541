"""The sampler's conditioning of several steps at a time."""

import pytest
import torch


# one step, the last ones fewer than the others, all in one; a token count that makes 128-column strips' rows ragged
@pytest.mark.gpu
@pytest.mark.parametrize("tokens,levels", [(1, 1), (12, 3), (100, 8), (101, 7), (400, 2)])
def test_rows_are_each_level_s_own(gpu_pkg, tokens, levels):
    """Every row's sums are taken in one order, whatever kernel its number of rows leads to."""
    with torch.device("cuda"):
        head = gpu_pkg.nn.DiffusionHead(use_batch_infer=True)
    cond = torch.randn(levels, tokens, 384, generator=torch.Generator(device="cuda").manual_seed(tokens), device="cuda")
    steps = head.step_conditioning(cond)
    assert len(steps) == levels
    for one, step in zip(cond, steps):
        alone = head.step_conditioning(one[None])[0]
        for got, want in zip(step, alone):
            assert got.is_contiguous() and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [0, 24, 36, 800])
def test_sampler(gpu_pkg, rows, monkeypatch):
    """The same positions however many steps are taken together, and from a head that is not as written."""
    from test_gpu_head import case, on_gpu

    g, batch, p, emb, pos, head = case(gpu_pkg, 12, 2, seed=5, samples=2)
    gb, ge = batch.to("cuda"), on_gpu(emb)
    rots = torch.stack([gpu_pkg.nn.diffusion_head.random_rotation(g, "cpu") for _ in range(5)]).cuda()
    sampler = gpu_pkg.nn.DiffusionSampler(head, num_samples=2, diffusion_steps=5)
    run = lambda: sampler(gb, ge, positions=pos.float().cuda(), rotations=rots, translations=rots[:, 0])["atom_positions"]
    seen, step_conditioning = [], head.step_conditioning
    monkeypatch.setattr(gpu_pkg.nn.diffusion_head, "STEP_ROWS", rows)
    monkeypatch.setattr(head, "step_conditioning", lambda c: (seen.append(len(c)), step_conditioning(c))[1])
    got = run()
    assert seen == {0: [], 24: [2, 2, 1], 36: [3, 2], 800: [5]}[rows]
    hook = head.register_forward_hook(lambda *a: None)
    want = run()
    hook.remove()
    assert len(seen) == {0: 0, 24: 3, 36: 2, 800: 1}[rows] and torch.equal(got, want)
