"""The transition of rows of 384 fp32 channels in one kernel (row_transition.hip)."""

import pytest
import torch


def _module(pkg, factor, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        mod = pkg.nn.DiffusionTransition(c_x=384, c_single_cond=None, num_intermediate_factor=factor)
    with torch.no_grad():
        for name, p in mod.named_parameters():
            p.normal_(0.0, 0.05, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    mod.invalidate()
    return mod


def _exact(mod, x):
    x = x.double()
    norm = mod.adaptive_layernorm.layer_norm
    y = torch.nn.functional.layer_norm(x, (384,), norm.weight.double(), norm.bias.double())
    a, b = (y @ mod.transition1.weight.bfloat16().double().T).chunk(2, dim=-1)
    return x + (torch.nn.functional.silu(a) * b) @ mod.adaptive_zero_init.transition2.weight.bfloat16().double().T


def _by_parts(pkg, mod, x):
    norm, p = mod.adaptive_layernorm.packed(), mod.packed()
    h = pkg.ops.linear(pkg.ops.layer_norm(x, norm["ln_w"], norm["ln_b"]), p["w1"], mode=pkg.lib.LINEAR_SWIGLU)
    return mod.adaptive_zero_init.run(h, None, x.dtype, residual=x.clone())


# a row; the edges of a tile of 64 and of its blocks of 32; more tiles than CUs; one chunk of hidden units and twice as many as usual
@pytest.mark.gpu
@pytest.mark.parametrize("rows,factor", [(1, 2), (31, 2), (33, 1), (63, 2), (64, 4), (65, 2), (257, 2), (16500, 2)])
def test_as_exact_as_three_kernels(gpu_pkg, rows, factor):
    """Rounded at the same places, fp32 sums of another order: few roundings to bf16 fall on the other side.  Against 64 bits the error
    is therefore that of the separate kernels: by root mean square up to a flip of some values in a hundred, 5 % (10 % for the 384
    values of one row); the largest by one flip more, a half."""
    mod = _module(gpu_pkg, factor, rows)
    x = torch.randn(rows, 384, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda")
    want, parts = _exact(mod, x), _by_parts(gpu_pkg, mod, x)
    norm = mod.adaptive_layernorm.packed()
    got = gpu_pkg.ops.row_transition(x.clone(), norm["ln_w"], norm["ln_b"], mod.packed()["w1_frags"],
                                     mod.adaptive_zero_init.packed()["w_frags"])
    e, ref = (got.double() - want).abs(), (parts.double() - want).abs()
    assert e.pow(2).mean().sqrt() <= (1.10 if rows == 1 else 1.05) * ref.pow(2).mean().sqrt()
    assert e.max() <= 1.5 * ref.max()


# the last size by parts, the first in one kernel; a batch of levels; a row behind the last is not written
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [8191, 8192, 8193])
def test_route(gpu_pkg, rows, monkeypatch):
    mod = _module(gpu_pkg, 2, 1)
    x = torch.randn(rows + 1, 384, generator=torch.Generator(device="cuda").manual_seed(rows), device="cuda")
    parts = _by_parts(gpu_pkg, mod, x[:rows].clone())
    seen = []
    one = gpu_pkg.ops.row_transition
    monkeypatch.setattr(gpu_pkg.ops, "row_transition", lambda *a: (seen.append(1), one(*a))[1])
    y = x.clone()
    got = mod.run(y[:rows], None, residual=True)
    assert got.data_ptr() == y.data_ptr() and len(seen) == (rows >= 8192)
    assert torch.equal(y[rows], x[rows])
    assert (got - parts).abs().max() <= 0.02 * parts.abs().max()
    # a result that is not added, another type: by parts
    mod.run(x[:rows], None, residual=False)
    mod.run(x[:rows].bfloat16(), None, residual=True)
    assert len(seen) == (rows >= 8192)


# layers of another width put in their place
@pytest.mark.gpu
def test_other_widths(gpu_pkg):
    mod = _module(gpu_pkg, 2, 2)
    mod.transition1, mod.adaptive_zero_init.transition2 = torch.nn.Linear(384, 1600, bias=False), torch.nn.Linear(800, 384, bias=False)
    mod.cuda()
    x = torch.randn(8192, 384, device="cuda")
    want = _exact(mod, x)
    assert (mod.run(x, None, residual=True) - want).abs().max() <= 0.02 * want.abs().max()


def test_refused(pkg):
    lib = pkg.lib.load()
    assert lib.af3_row_transition_forward(None, None, None, None, None, 768, 64, None) == -1
