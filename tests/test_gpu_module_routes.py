"""Runs of modules that go to the library as one call, against the same modules one by one: what a user has put between
them (forward hooks, a sub-module of another class) has its effect, and the results are the ones of the single call."""

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def on_gpu(mod, std=0.05):
    g = torch.Generator().manual_seed(1)
    for p in mod.parameters():
        p.data.normal_(0.0, std, generator=g)
    return mod.to("cuda:0")


def counter(mod, seen):
    return mod.register_forward_hook(lambda m, args, out: seen.append(m))


def trunk_inputs(n=37):
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    mask = (torch.arange(n, device="cuda") < n - 3).float()
    return rnd(n, n, 128), (mask[:, None] * mask[None, :]).contiguous(), rnd(n, 384), mask


def test_hooks_in_a_pairformer_stack(gpu_pkg):
    stack = on_gpu(gpu_pkg.nn.PairformerStack(num_blocks=3))
    pair, pm, single, sm = trunk_inputs()
    run = lambda: stack(pair.clone(), pm, single.clone(), sm)
    want, blocks, seen = run(), stack.trunk_pairformer, []
    for where, count in ((blocks[1], 1), (blocks[2].single_attention_.adaptive_layernorm, 1), (None, 3)):
        seen.clear()
        if where is None:
            every = lambda m, args, out: seen.append(m) if isinstance(m, gpu_pkg.nn.PairformerBlock) else None
            hook = torch.nn.modules.module.register_module_forward_hook(every)
        else:
            hook = counter(where, seen)
        got = run()
        hook.remove()
        assert len(seen) == count
        # (module by module the single track's products sum in another order: bf16 roundings of an update of order one)
        assert torch.equal(got[0], want[0]) and float((got[1] - want[1]).norm() / want[1].norm()) < 1e-2
    assert all(torch.equal(a, b) for a, b in zip(run(), want))


def test_a_sub_module_of_another_class(gpu_pkg):
    class Doubled(gpu_pkg.nn.Transition):
        def run(self, x, residual):
            return super().run(super().run(x, residual), residual)

    blk = on_gpu(gpu_pkg.nn.PairformerBlock(with_single=False))
    pair, pm, _, _ = trunk_inputs()
    want = blk.pair_transition.run(blk(pair.clone(), pm), True)
    other = Doubled(c_x=128)
    other.load_state_dict(blk.pair_transition.state_dict())
    blk.pair_transition = other.to("cuda:0")
    assert torch.equal(blk(pair.clone(), pm), want)


def test_hooks_in_a_run_of_evoformer_blocks(gpu_pkg):
    blocks, seen = [on_gpu(gpu_pkg.nn.EvoformerBlock()) for _ in range(2)], []
    pair, pm, _, sm = trunk_inputs(19)
    msa = torch.randn(5, 19, 64, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda")
    run = lambda: gpu_pkg.nn.evoformer.evoformer_loop(blocks, msa.clone(), pair.clone(), sm.expand(5, -1).contiguous(), pm)
    want = run()
    hook = counter(blocks[1], seen)
    got = run()
    hook.remove()
    assert len(seen) == 1 and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def diffusion_case(pkg, n):
    mod = on_gpu(pkg.nn.DiffusionTransformer(num_blocks=4, super_block_size=2))
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    act, cond, pair = rnd(2, n, 768).bfloat16(), rnd(n, 384), rnd(n, n, 128)
    mask = (torch.arange(n, device="cuda") < n - 3).float()
    return mod, mask, lambda mask=mask, **k: mod(act.clone(), mask, cond, pair, **k)


@pytest.mark.parametrize("n", [24, 21])       # pair logits in quads of keys, and in rows
def test_hooks_in_a_diffusion_transformer(gpu_pkg, n):
    (mod, _, run), seen = diffusion_case(gpu_pkg, n), []
    want = run()
    hook = counter(mod.self_attention[1].adaptive_layernorm, seen)
    got = run()
    hook.remove()
    assert len(seen) == 1 and torch.equal(got, want)


# the windows' kernel with quads of keys outermost, the order the model gives it, against rows of keys: a window of one
# query, shorter than a tile of 64 keys, just past it, full; more windows than two on every CU
@pytest.mark.parametrize("samples,s,q,k", [(2, 3, 32, 128), (2, 5, 7, 60), (1, 2, 1, 4), (3, 4, 31, 64), (1, 4, 32, 68), (3, 171, 32, 128),
                                           (1, 600, 9, 60), (2, 3, 8, 61)])
def test_hooks_in_an_atom_transformer(gpu_pkg, samples, s, q, k):
    mod, seen = on_gpu(gpu_pkg.nn.DiffusionCrossAttTransformer()), []
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    idx = torch.randint(0, s * q, (s, k), generator=g, device="cuda")
    gather = (idx, torch.rand(s, k, generator=g, device="cuda") > 0.2)
    act, mk = rnd(samples, s, q, 128).bfloat16(), gather[1].float()
    mq = (torch.rand(s, q, generator=g, device="cuda") > 0.2).float()
    sq = rnd(s, q, 128)
    sk = sq.view(s * q, 128)[idx] * gather[1][..., None]
    cond = mod.conditioning(sq, sk, rnd(s, q, k, 16), keys_are_query_atoms=gather)
    assert cond[0].dim() == (6 if k % 4 == 0 else 5)
    run = lambda: mod(act.clone(), mq, gather, mk, sq, sk, None, cond=cond)
    want = run()
    hook = counter(mod.cross_attention[1].k_adaptive_layernorm, seen)
    got = run()
    hook.remove()
    assert len(seen) == 1 and torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("n", [24, 21])
def test_a_key_mask_per_sample(gpu_pkg, n):
    _, mask, run = diffusion_case(gpu_pkg, n)
    other = mask.roll(5)
    got = run(torch.stack([mask, other]))
    assert torch.equal(got[0], run()[0]) and torch.equal(got[1], run(other)[1]) and not torch.equal(got[1], run()[1])


@pytest.mark.parametrize("n", [24, 21])
def test_pair_logits_of_another_type_or_order(gpu_pkg, n):
    """Logits that a caller has computed and kept: bf16, a strided view, rows for one super-block and quads for the other."""
    mod, _, run = diffusion_case(gpu_pkg, n)
    pair = torch.randn(n, n, 128, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    logits = mod.pair_logits(pair)
    want = run(pair_logits=logits)
    strided = [torch.stack([t, -t], dim=-1)[..., 0] for t in logits]
    assert not strided[0][0].is_contiguous() and torch.equal(run(pair_logits=strided), want)
    half = [t.bfloat16() for t in logits]
    assert torch.equal(run(pair_logits=half), run(pair_logits=[t.float() for t in half]))
    if n % 4 == 0:
        rows = logits[0].transpose(-3, -2).reshape(*logits[0].shape[:2], n, n)
        assert torch.equal(run(pair_logits=[rows, logits[1]]), want)


def test_a_later_block_with_a_wider_single_transition(gpu_pkg):
    """The scratch is one for all blocks of a run."""
    n, blocks = 37, [on_gpu(gpu_pkg.nn.PairformerBlock()) for _ in range(3)]
    blocks[1].single_transition = on_gpu(gpu_pkg.nn.Transition(c_x=384, num_intermediate_factor=9))
    pair, pm, single, sm = trunk_inputs(n)
    one = pair.clone(), single.clone()
    for blk in blocks:
        one = blk(one[0], pm, one[1], sm)
    gpu_pkg.ops.release_workspaces()
    two = gpu_pkg.nn.pairformer_loop(blocks, pair.clone(), pm, single.clone(), sm)
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])


def test_an_msa_mask_that_broadcasts(gpu_pkg):
    """One mask row for all MSA rows: what the attention takes from the mask is its maximum over the rows."""
    att = on_gpu(gpu_pkg.nn.MSAAttention())
    pair, _, _, mask = trunk_inputs(19)
    msa = torch.randn(5, 19, 64, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda")
    want, got = att(msa, mask.expand(5, -1).contiguous(), pair), att(msa, mask[None], pair)
    assert float((got - want).norm() / want.norm()) < 1e-2      # (bf16 products and sums in another order)


def test_a_batch_of_single_representations(gpu_pkg):
    stack = on_gpu(gpu_pkg.nn.PairformerStack(num_blocks=2))
    pair, pm, single, sm = trunk_inputs()
    both = torch.stack([single, single.roll(3, 0)])
    got = stack(pair.clone(), pm, both.clone(), torch.stack([sm, sm]))
    for i in range(2):
        want = stack(pair.clone(), pm, both[i].clone(), sm)
        # (a single sequence's products may sum in another order)
        assert torch.equal(got[0], want[0]) and float((got[1][i] - want[1]).norm() / want[1].norm()) < 1e-2


def test_modules_left_on_the_cpu_are_refused(gpu_pkg):
    nn = gpu_pkg.nn
    pair, pm, single, sm = trunk_inputs(12)
    msa, act, cond = torch.zeros(3, 12, 64, device="cuda"), torch.zeros(1, 12, 768, device="cuda"), torch.zeros(12, 384, device="cuda")
    logits = [torch.zeros(1, 16, 3, 12, 4, device="cuda")]
    for call in (lambda: nn.PairformerBlock()(pair, pm, single, sm), lambda: nn.PairformerStack(num_blocks=2)(pair, pm, single, sm),
                 lambda: nn.EvoformerBlock()(msa, pair, sm.expand(3, -1).contiguous(), pm),
                 lambda: nn.OuterProductMean()(msa, sm.expand(3, -1).contiguous()),
                 lambda: nn.MSAAttention()(msa, sm.expand(3, -1).contiguous(), pair),
                 lambda: nn.DiffusionTransformer(num_blocks=1, super_block_size=1)(act, sm, cond, pair, pair_logits=logits)):
        with pytest.raises(ValueError, match="cpu"):
            call()


@pytest.mark.parametrize("n", [1, 5, 33, 66, 67, 129, 259])
def test_single_attention_over_a_partly_filled_quad(gpu_pkg, n):
    """The bias of the last keys, where their quad is partly filled, decides most of a row's softmax: logits of +- 6 from
    the pair tensor, and the last three keys 4 above the others.  Module by module the bias comes in rows."""
    blk, seen = on_gpu(gpu_pkg.nn.PairformerBlock()), []
    blk.single_pair_logits_projection.weight.data.zero_()[:, :3] = torch.tensor([4.0, 3.0, 2.0])
    blk.single_pair_logits_norm.weight.data.fill_(1.0)
    for m in (blk.triangle_multiplication_outgoing, blk.triangle_multiplication_incoming, blk.pair_attention1, blk.pair_attention2):
        m.output_projection.weight.data.zero_()
    blk.pair_transition.transition2.weight.data.zero_()
    blk.invalidate()
    pair, _, single, _ = trunk_inputs(n)
    pair[:, max(0, n - 3):, 0] += 1.0
    pm, sm = torch.ones(n, n, device="cuda"), (torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda") > 0.2).float()
    sm[-1] = 1.0
    run = lambda: blk(pair.clone(), pm, single.clone(), sm)[1] - single
    got = run()
    hook = counter(blk.single_attention_.adaptive_layernorm, seen)
    want = run()
    hook.remove()
    # fp32 sums of products in another order, rounded to bf16 once: an ulp here and there
    assert len(seen) == 1 and float((got - want).norm() / want.norm()) < 2.0 ** -9


def test_single_calls_under_capture(gpu_pkg):
    """Each captured once and replayed on new contents, with the program's own work between the replays.  (One eager call
    first, as for any capture: it packs the weights and grows the scratch.)"""
    nn = gpu_pkg.nn
    stack, blocks = on_gpu(nn.PairformerStack(num_blocks=3)), [on_gpu(nn.EvoformerBlock()) for _ in range(2)]
    pair, pm, single, sm = trunk_inputs()
    msa, mm = torch.randn(5, 37, 64, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda"), sm.expand(5, -1).contiguous()
    act, cond = msa.new_empty(2, 37, 768).normal_().bfloat16(), single.clone()
    transformer = on_gpu(nn.DiffusionTransformer(num_blocks=2, super_block_size=1))
    logits = transformer.pair_logits(pair)

    def trunk(p, s):
        return stack(p.clone(), pm, s.clone(), sm)

    def evoformer(p, m):
        return nn.evoformer.evoformer_loop(blocks, m.clone(), p.clone(), mm, pm)

    def diffusion(a, c):
        return (transformer(a.clone(), sm, c, pair, pair_logits=logits),)

    for fn, inputs in ((trunk, (pair, single)), (evoformer, (pair, msa)), (diffusion, (act, cond))):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            fn(*inputs)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = fn(*inputs)
        for i in range(3):
            for t in inputs:
                t.mul_(-1.0).add_(0.125 * i)
            want = fn(*inputs)
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, want)), (fn.__name__, i)


def test_two_threads_on_one_stream(gpu_pkg):
    """Their runs of blocks share the stream's scratch: one is enqueued whole, then the other."""
    stack = on_gpu(gpu_pkg.nn.PairformerStack(num_blocks=3))
    stack.load_hip_params()
    cases = [trunk_inputs(n) for n in (37, 50)]
    run = lambda c: stack(c[0].clone(), c[1], c[2].clone(), c[3])
    want, got = [run(c) for c in cases], [[], []]
    start = threading.Barrier(2)

    def work(i):
        start.wait()
        for _ in range(20):
            got[i].append(run(cases[i]))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 20 and all(torch.equal(a, b) for out in got[i] for a, b in zip(out, want[i]))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,factor", [(1, 2), (127, 1), (128, 2), (129, 2), (1700, 4), (120001, 2)])
@pytest.mark.parametrize("residual", [True, False])
def test_unconditioned_transition_in_one_kernel(gpu_pkg, rows, factor, residual):
    """128 channels without conditioning: the bits of the LayerNorm and the two products, which a tensor off 16 bytes takes."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    with torch.device("cuda"):
        mod = gpu_pkg.nn.DiffusionTransition(c_x=128, c_single_cond=None, num_intermediate_factor=factor)
    with torch.no_grad():
        for name, p in mod.named_parameters():
            p.normal_(0.0, 0.1, generator=g)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    mod.invalidate()
    x = torch.randn(rows, 128, generator=g, device="cuda") * 3 + 1
    got = mod.run(x.clone(), None, residual=residual)
    norm = mod.adaptive_layernorm.packed()
    h = gpu_pkg.ops.linear(gpu_pkg.ops.layer_norm(x, norm["ln_w"], norm["ln_b"]), mod.packed()["w1"], mode=gpu_pkg.lib.LINEAR_SWIGLU)
    want = mod.adaptive_zero_init.run(h, None, x.dtype, residual=x.clone() if residual else None)
    assert got.dtype == torch.float32 and torch.isfinite(got).all() and torch.equal(got, want) and not torch.equal(got, x)
