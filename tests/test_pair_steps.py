"""The pair operators at few tokens, a run of them in one kernel (pair_step.hip), against one kernel per operator."""

import pytest
import torch


def _block(pkg, c=128, factor=4, seed=0, device="cuda", std=0.05, heads=16):
    """A block with random weights: LayerNorm weights around 1, everything else N(0, std)."""
    gen = torch.Generator(device=device).manual_seed(seed)
    with torch.device(device):
        blk = pkg.nn.PairformerBlock(c_pair=c, num_intermediate_factor=factor, with_single=c == 128, n_heads=heads,
                                     c_single=24 * heads)
    with torch.no_grad():
        for name, p in blk.named_parameters():
            p.normal_(0.0, std, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    blk.invalidate()
    return blk


def _inputs(n, c, io, padding, seed=1, heads=16):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    seq = (torch.arange(n, device="cuda") < n - padding).float()
    pair = torch.randn(n, n, c, generator=gen, device="cuda").to(io)
    single = torch.randn(n, 24 * heads, generator=gen, device="cuda").to(io)
    return pair, (seq[:, None] * seq[None, :]).contiguous(), single, seq


def _run(blk, pair, mask, single, seq):
    out = blk(pair.clone(), mask, single.clone(), seq) if blk.with_single else (blk(pair.clone(), mask),)
    torch.cuda.synchronize()
    return out


def _run_general(blk, *inputs):
    s = blk.native()
    held, s.pair_frags, s.pair_channels = (s.pair_frags, s.pair_channels), None, 128
    try:
        return _run(blk, *inputs)
    finally:
        s.pair_frags, s.pair_channels = held


# sizes: one pixel; rows shorter than a group of 16 positions, one longer; tiles that cross rows and that do not; a key tile
# of 64 and one more; the contraction's two kernels; both sizes of patches; the largest.  Hidden layers of one chunk, a part
# of one and two; more than one block of 32 heads.
CASES = [(1, 128, 4, 16, 0), (7, 128, 4, 16, 2), (16, 128, 4, 16, 0), (17, 128, 4, 40, 3), (33, 128, 1, 16, 0), (63, 128, 4, 16, 5),
         (64, 128, 2, 16, 0), (65, 128, 4, 16, 30), (127, 128, 4, 16, 0), (129, 128, 3, 16, 11), (208, 128, 4, 16, 9),
         (24, 96, 1, 16, 3), (90, 96, 4, 16, 1),
         (209, 128, 4, 16, 9), (217, 96, 2, 16, 0), (398, 128, 2, 16, 29),
         # a transition in tiles of 32 and 64 positions, by the rounds they make; the incoming product's step and its two kernels;
         # the last sizes of a bf16 stream, and one that only an fp32 stream takes in steps
         (152, 128, 4, 16, 7), (153, 128, 4, 16, 0), (176, 128, 1, 40, 5), (177, 128, 4, 16, 11), (193, 128, 2, 16, 0),
         (493, 128, 4, 16, 17), (545, 96, 4, 16, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,factor,heads,padding", CASES)
def test_steps_give_the_bits_of_one_kernel_per_operator(gpu_pkg, n, c, factor, heads, padding, io):
    """The same sums in the same order, rounded at the same places."""
    blk, inputs = _block(gpu_pkg, c, factor, n, heads=heads), _inputs(n, c, io, padding, heads=heads)
    got, want = _run(blk, *inputs), _run_general(blk, *inputs)
    for x, y, before in zip(got, want, (inputs[0], inputs[2])):
        assert torch.isfinite(x).all() and not torch.equal(x, before) and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,factor,padding", [(154, 128, 4, 0), (160, 128, 4, 9), (162, 96, 4, 3), (163, 128, 4, 0)])
def test_projections_four_workgroups_to_a_cu(gpu_pkg, n, c, factor, padding, io):
    """The first and the last sizes of that form, a short last tile, and one size past them."""
    blk, inputs = _block(gpu_pkg, c, factor, n), _inputs(n, c, io, padding)
    got, want = _run(blk, *inputs), _run_general(blk, *inputs)
    for x, y, before in zip(got, want, (inputs[0], inputs[2])):
        assert torch.isfinite(x).all() and not torch.equal(x, before) and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,factor,padding", [(1, 2, 0), (7, 2, 2), (16, 1, 0), (17, 2, 3), (33, 2, 0), (64, 1, 5), (65, 2, 30),
                                              (127, 2, 0), (129, 1, 9), (187, 2, 11), (208, 2, 0), (301, 2, 11), (515, 2, 40)])
def test_64_channels_as_they_are(gpu_pkg, n, factor, padding, io):
    """Kernels for 64 channels against the 128-channel ones on the zero-padded tensor: the same products and roundings, only
    the LayerNorms' sums of the padded form carry 64 times the square of a mean that they take out again.  A statistic that
    is an fp32 rounding away moves few bf16 values by one place, 2^-8 of the value."""
    blk, inputs = _block(gpu_pkg, 64, factor, n), _inputs(n, 64, io, padding)
    assert blk.native().pair_channels == 64
    got, want, before = _run(blk, *inputs)[0], _run_general(blk, *inputs)[0], inputs[0].double()
    assert got.dtype == io and torch.isfinite(got).all()
    diff, update = got.double() - want.double(), want.double() - before
    assert update.square().mean() > 0
    assert diff.square().mean().sqrt() <= 2.0 ** -8 * update.square().mean().sqrt()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [33, 150, 301])
def test_64_channels_far_from_zero(gpu_pkg, n):
    """Attention logits in the hundreds: the softmax moves its base, and tiles taken without a look at their maximum are
    repeated.  One bf16 place of one of 64 channels moves such a logit by 10 / 2^8, and a probability by 4 %; few differ."""
    blk, inputs = _block(gpu_pkg, 64, 2, n), _inputs(n, 64, torch.bfloat16, 3)
    with torch.no_grad():
        for att in (blk.pair_attention1, blk.pair_attention2):
            att.pair_bias_projection.weight *= 200.0
    blk.invalidate()
    got, want, before = _run(blk, *inputs)[0], _run_general(blk, *inputs)[0], inputs[0].double()
    assert torch.isfinite(got).all()
    diff, update = got.double() - want.double(), want.double() - before
    assert diff.square().mean().sqrt() <= 2.0 ** -6 * update.square().mean().sqrt()


@pytest.mark.gpu
def test_64_channels_that_are_padded_after_all(gpu_pkg):
    """Blocks the 64-channel kernels do not take; and a tensor that does not begin on 16 bytes, which is copied."""
    blk, (pair, mask, _, _) = _block(gpu_pkg, 64, 2, 5), _inputs(40, 64, torch.bfloat16, 3)
    want = blk(pair.clone(), mask)
    store = torch.empty(pair.numel() + 1, dtype=pair.dtype, device="cuda")
    odd = store[1:].view(pair.shape).copy_(pair)
    got = blk(odd, mask)
    assert got.data_ptr() == odd.data_ptr() and (got.float() - want.float()).square().mean() < 1e-4 * want.float().square().mean()
    wide = _block(gpu_pkg, 64, 4, 5)
    assert wide.native().pair_channels == 128
    assert torch.isfinite(wide(pair.clone(), mask)).all()


@pytest.mark.gpu
def test_64_channels_past_the_last_size_of_their_kernels(gpu_pkg, monkeypatch):
    """Padded, by a structure of its own: the bits of the 128-channel kernels (the last size made small)."""
    blk, inputs = _block(gpu_pkg, 64, 2, 5), _inputs(40, 64, torch.bfloat16, 3)
    want = _run_general(blk, *inputs)[0]
    assert not torch.equal(_run(blk, *inputs)[0], want)
    monkeypatch.setattr(gpu_pkg.lib, "PAIR64_MAX_TOKENS", 39)
    assert torch.equal(_run(blk, *inputs)[0], want) and blk.native().pair_channels == 64


@pytest.mark.gpu
@pytest.mark.parametrize("io", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [9, 150])
def test_64_channels_at_any_address(gpu_pkg, n, io):
    """The bits do not depend on where the tensor begins."""
    blk, (pair, mask, _, _) = _block(gpu_pkg, 64, 2, n), _inputs(n, 64, io, 2)
    want = blk(pair.clone(), mask)
    store = torch.full((pair.numel() + 5,), 7.0, dtype=io, device="cuda")
    odd = store[3:-2].view(pair.shape).copy_(pair)
    got = blk(odd, mask)
    assert want.data_ptr() % 16 == 0 and odd.data_ptr() % 16 and got.data_ptr() == odd.data_ptr() and torch.equal(got, want)
    assert (store[:3] == 7.0).all() and (store[-2:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n,count", [(5, 3), (48, 19), (130, 10)])
def test_a_run_of_blocks_is_its_blocks_one_by_one(gpu_pkg, n, count):
    """The last step of a block makes the next block's first operands, and the buffers of the pair logits come round again
    after eight blocks: the same bits as a call per block."""
    blocks, inputs = [_block(gpu_pkg, seed=i) for i in range(count)], _inputs(n, 128, torch.bfloat16, 2)
    pair, mask, single, seq = inputs
    got = gpu_pkg.nn.pairformer_loop(blocks, pair.clone(), mask, single.clone(), seq)
    want = (pair, single)
    for blk in blocks:
        want = _run(blk, want[0], mask, want[1], seq)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.gpu
def test_incoming_mask_of_its_own(gpu_pkg):
    """An Evoformer block gives the incoming product the transposed mask: one that is not symmetric."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    n, rows = 43, 9
    with torch.device("cuda"):
        blk = gpu_pkg.nn.EvoformerBlock()
    with torch.no_grad():
        for name, p in blk.named_parameters():
            p.normal_(0.0, 0.05, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    blk.invalidate()
    pair, msa = torch.randn(n, n, 128, generator=gen, device="cuda"), torch.randn(rows, n, 64, generator=gen, device="cuda")
    mask, msa_mask = (torch.rand(n, n, generator=gen, device="cuda") > 0.3).float(), torch.ones(rows, n, device="cuda")
    got = blk(msa.clone(), pair.clone(), msa_mask, mask)[1]
    s = blk.native()
    frags, s.pair.pair_frags = s.pair.pair_frags, None
    want = blk(msa.clone(), pair.clone(), msa_mask, mask)[1]
    s.pair.pair_frags = frags
    assert torch.equal(got, want)


def test_fragment_order(pkg):
    """[row / 32][column / 16][(column / 8) % 2][row % 32][column % 8]; exchanged rows are their own inverse."""
    base = pkg.nn.base
    w = torch.arange(64 * 48).reshape(64, 48)
    f = base.fragments(w).reshape(2, 3, 2, 32, 8)
    for r in (0, 5, 31, 32, 63):
        for c in (0, 7, 8, 15, 16, 47):
            assert f[r // 32, c // 16, c // 8 % 2, r % 32, c % 8] == w[r, c]
    g = base.fragments(w, swap23=True).reshape(2, 3, 2, 32, 8)
    assert torch.equal(g[:, :, :, 4], f[:, :, :, 8]) and torch.equal(g[:, :, :, 27], f[:, :, :, 23]) and torch.equal(g[:, :, :, 3], f[:, :, :, 3])


@pytest.mark.parametrize("factor,rows", [(4, 2880 + 1536 + 32), (2, 2880 + 768 + 32)])
def test_all_matrices_of_a_block_are_in_its_fragments(pkg, factor, rows):
    blk = _block(pkg, factor=factor, device="cpu")
    s = blk.native()
    frags = blk._native[2]
    assert s.pair_frags == frags.data_ptr() and frags.dtype == torch.bfloat16 and frags.numel() == rows * 128
    q = blk.pair_attention1.packed()["w_qkvg"]
    assert torch.equal(frags[:128 * 128], pkg.nn.base.fragments(q[0], swap23=True))
    at = 768 * 128      # the matrices in their own order of rows, up to the transition's second
    for w in (blk.triangle_multiplication_outgoing.packed()["w_gl"], blk.triangle_multiplication_outgoing.packed()["w_out"]):
        assert torch.equal(frags[at:at + 128 * 128], pkg.nn.base.fragments(w))
        at += 128 * 128
    w2 = blk.pair_transition.packed()["w2"]
    assert torch.equal(frags[-w2.numel():], pkg.nn.base.fragments(w2))
    assert torch.equal(frags[-w2.numel() - 32 * 128:-w2.numel()], pkg.nn.base.fragments(blk.packed()["w_logits"]))


@pytest.mark.gpu
@pytest.mark.parametrize("n,blocks", [(40, 1), (40, 2), (40, 3), (33, 11), (133, 5), (145, 4)])
def test_stacks_give_the_bits_of_their_blocks(gpu_pkg, n, blocks):
    """The streams of a stack meet for one or two blocks at a time, and more blocks than the eight buffers of pair logits go round."""
    run = [_block(gpu_pkg, seed=i) for i in range(blocks)]
    pair, mask, single, seq = _inputs(n, 128, torch.bfloat16, 3)
    want = (pair.clone(), single.clone())
    for blk in run:
        want = blk(*want[:1], mask, want[1], seq)
    for _ in range(3):
        got = gpu_pkg.nn.pairformer_loop(run, pair.clone(), mask, single.clone(), seq)
        assert all(torch.isfinite(x).all() and torch.equal(x, y) for x, y in zip(got, want))
