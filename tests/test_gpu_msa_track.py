"""The MSA track's own kernels (64 channels) at the edges of their tiles of 32 and 64 positions, against the float64
oracle: fewer MSA rows or tokens than a tile, one more, counts that are no multiple of 8, masks that are not 0 or 1, both
stream types; and a run of blocks in one call against the same blocks one by one."""

import pytest
import torch

from oracle import af3_msa_oracle as M
from oracle import af3_oracle as O

pytestmark = pytest.mark.gpu
D = torch.float64


def compare(name, got, want, rms_tol=1e-2, max_tol=8e-2):
    got, want = got.double().cpu(), want.double()
    scale = float((want ** 2).mean().sqrt())
    rms, mx = float(((got - want) ** 2).mean().sqrt()) / scale, float((got - want).abs().max()) / scale
    print(f"{name}: rms {rms:.3e} max {mx:.3e}", flush=True)
    assert torch.isfinite(got).all() and rms <= rms_tol and mx <= max_tol, (name, rms, mx)


def inputs(rows, n):
    g = torch.Generator().manual_seed(1000 * rows + n)
    p = {k: O.round_bf16(v) for k, v in M.make_evoformer_block_params(g, std=0.05).items()}
    msa, pair = O.round_bf16(torch.randn(rows, n, 64, generator=g)), O.round_bf16(torch.randn(n, n, 128, generator=g))
    mask = O.round_bf16(torch.rand(rows, n, generator=g) * 0.9 + 0.1) * (torch.rand(rows, n, generator=g) > 0.2)
    mask[0] = 1
    return p, msa, pair, mask


@pytest.mark.parametrize("rows,n", [(1, 9), (8, 8), (33, 65), (65, 130), (129, 31), (300, 7)])
def test_msa_operators(gpu_pkg, rows, n):
    p, msa, pair, mask = inputs(rows, n)
    for name, cls, ref in (
            ("outer_product_mean", "OuterProductMean", lambda q: M.outer_product_mean(msa.double(), mask.double(), q)),
            ("msa_attention1", "MSAAttention", lambda q: M.msa_attention(msa.double(), mask.double(), pair.double(), q))):
        mod = getattr(gpu_pkg.nn, cls)()
        mod.load_state_dict(O._sub(p, name))
        mod.to("cuda:0")
        want = ref(O._sub(O.cast_params(p, D), name))
        args = (mask.to("cuda:0"),) + ((pair.to("cuda:0"),) if cls == "MSAAttention" else ())
        compare(f"{cls} {rows} {n}", mod(msa.to("cuda:0"), *args), want)
        compare(f"{cls} {rows} {n} bf16", mod(msa.to("cuda:0").bfloat16(), *args), want, 1.2e-2)


@pytest.mark.parametrize("rows", [1, 31, 33, 5000])
@pytest.mark.parametrize("factor", [1, 2, 4])
def test_transition_of_narrow_rows(gpu_pkg, rows, factor):
    g = torch.Generator().manual_seed(rows + factor)
    p = {k: O.round_bf16(v) for k, v in O.make_transition_params(g, 64, factor, std=0.1).items()}
    x = O.round_bf16(torch.randn(rows, 64, generator=g))
    mod = gpu_pkg.nn.Transition(c_x=64, num_intermediate_factor=factor)
    mod.load_state_dict(p)
    mod.to("cuda:0")
    compare(f"transition {rows} {factor}", mod(x.to("cuda:0")), O.transition(x.double(), O.cast_params(p, D)))


@pytest.mark.parametrize("rows,n,dtype", [(40, 33, torch.bfloat16), (9, 70, torch.float32)])
def test_a_run_of_blocks_is_the_blocks_in_turn(gpu_pkg, rows, n, dtype):
    _, msa, pair, mask = inputs(rows, n)
    blocks = []
    for i in range(3):
        blk = gpu_pkg.nn.EvoformerBlock()
        g = torch.Generator().manual_seed(i)
        blk.load_state_dict({k: O.round_bf16(v) for k, v in M.make_evoformer_block_params(g, std=0.05).items()})
        blocks.append(blk.to("cuda:0"))
    pair_mask = (torch.rand(n, n, generator=torch.Generator().manual_seed(n)) > 0.2).float().to("cuda:0")
    t = lambda x: x.to("cuda:0").to(dtype)
    one, two = (t(msa), t(pair)), (t(msa), t(pair))
    for blk in blocks:
        one = blk(*one, mask.to("cuda:0"), pair_mask)
    two = gpu_pkg.nn.evoformer.evoformer_loop(blocks, *two, mask.to("cuda:0"), pair_mask)
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1])


@pytest.mark.parametrize("rows,n", [(16, 24), (12, 24), (16, 21)])       # operands produced transposed; by strided copies
@pytest.mark.parametrize("c", [32, 128])
def test_msa_operators_of_other_widths(gpu_pkg, c, rows, n):
    g = torch.Generator().manual_seed(c + rows + n)
    rb = lambda *s: O.round_bf16(torch.randn(*s, generator=g))
    msa, pair, mask = rb(rows, n, c), rb(n, n, 128), (torch.rand(rows, n, generator=g) > 0.2).float()
    mask[0] = 1
    for cls, args in (("OuterProductMean", (mask,)), ("MSAAttention", (mask, pair))):
        mod = getattr(gpu_pkg.nn, cls)(c_msa=c)
        for p in mod.parameters():
            p.data = O.round_bf16(torch.randn(p.shape, generator=g) * 0.1 + (1.0 if p.dim() == 1 else 0.0))
        q = {k: v.double() for k, v in mod.state_dict().items()}
        ref = M.outer_product_mean if cls == "OuterProductMean" else M.msa_attention
        want = ref(msa.double(), *(a.double() for a in args), q)
        assert not mod.native
        compare(f"{cls} {c} channels {rows} {n}", mod.to("cuda:0")(msa.to("cuda:0"), *(a.to("cuda:0") for a in args)), want)


@pytest.mark.parametrize("rows,n", [(33, 70), (9, 21)])
@pytest.mark.parametrize("poison", [float("nan"), float("inf")])
def test_a_masked_position_that_is_not_finite(gpu_pkg, rows, n, poison):
    """The mask multiplies, as in the reference: what is not finite stays so under a mask of zero, in the tokens and rows
    that it is part of (the last MSA row, which the tiles repeat behind the end, among them) and in no other."""
    p, msa, pair, mask = inputs(rows, n)
    for at in ((rows - 1, 3), (2, n - 1)):
        msa[at], mask[at] = poison, 0
    for name, cls, ref, more in (("outer_product_mean", "OuterProductMean", M.outer_product_mean, ()),
                                 ("msa_attention1", "MSAAttention", M.msa_attention, (pair,))):
        mod = getattr(gpu_pkg.nn, cls)()
        mod.load_state_dict(O._sub(p, name))
        mod.to("cuda:0")
        want = ref(msa.double(), mask.double(), *(x.double() for x in more), O._sub(O.cast_params(p, D), name))
        got = mod(*(x.to("cuda:0") for x in (msa, mask, *more))).cpu()
        lost = torch.isnan(want)
        assert torch.equal(torch.isnan(got), lost) and 0 < int(lost.sum()) < lost.numel() // 2
        compare(f"{cls} {rows} {n} {poison}", got[~lost], want[~lost])
