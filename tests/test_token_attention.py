"""Heads of 48 over plain keys (attention.hip, token_attention_kernel) against the general form of the same arithmetic."""

import pytest
import torch


# keys that fill no tile of 64, one, two and three of them, and a few past a tile; queries of one and of two tiles of 128; the mask
# over the end of a sequence, its first tile, single keys and a whole sequence
@pytest.mark.gpu
@pytest.mark.parametrize("batch,n,mask", [(1, 4, "end"), (3, 36, "some"), (2, 64, "none"), (5, 68, "end"), (2, 124, "first"), (1, 128, "all"),
                                          (2, 132, "some"), (1, 192, "first"), (5, 200, "end"), (2, 324, "some"), (1, 516, "first")])
def test_token_attention_gives_the_bits_of_the_general_form(gpu_pkg, batch, n, mask):
    """A bias that does not begin on 16 bytes takes the general form; both orders of an aligned one take the kernel."""
    g = torch.Generator(device="cuda").manual_seed(batch * n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, h = 768, 16
    x, w, qb = rnd(batch, n, c).bfloat16(), (rnd(4 * c, c) * 0.05).bfloat16(), rnd(c)
    logits = rnd(h, n, n) * 3
    logits[:, 0] += 40                                       # a row whose maximum moves the base
    logits[:, -1] *= 10
    keep = torch.ones(n, device="cuda")
    if mask == "end":
        keep[n - n // 8 - 1:] = 0
    elif mask == "first":
        keep[:70] = 0
    elif mask == "some":
        keep[::3] = 0
    elif mask == "all":
        keep[:] = 0
    off = torch.empty(logits.numel() + 1, device="cuda")[1:].view_as(logits)
    off.copy_(logits)
    run = lambda b: gpu_pkg.ops.batch_diffusion_self_attention(x, keep, b, w, qb, h, out_dtype=torch.float32)
    want = run(off)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    assert torch.equal(run(logits), want) and torch.equal(run(gpu_pkg.ops.quad_major_bias(logits)), want)
    one = gpu_pkg.ops.batch_diffusion_self_attention(x[:1].contiguous(), keep, logits, w, qb, h, out_dtype=torch.float32)
    assert torch.equal(one, run(logits).view(batch, n, c)[:1].reshape(one.shape))


@pytest.mark.gpu
@pytest.mark.parametrize("batch,shared,sq,sk", [(2, 1, 4, 4), (4, 2, 36, 68), (6, 3, 33, 36), (6, 1, 128, 200), (5, 5, 130, 64), (3, 1, 1, 132)])
def test_a_bias_that_batch_entries_share(gpu_pkg, batch, shared, sq, sk):
    """Cross-attention of heads of 48 without padding masks: entry b reads the logits b % shared, against float64 arithmetic on the
    projections as they are stored.  What is left are roundings to 8 bits (probabilities, a projection that falls on the other side of
    one): 1e-2 of the result's rms."""
    g = torch.Generator(device="cuda").manual_seed(100 * batch + sk)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, h = 192, 4
    q, m, qb = rnd(batch, sq, c).bfloat16(), rnd(batch, sk, c).bfloat16(), rnd(c)
    w_qg, w_kv = ((rnd(2 * c, c) * 0.07).bfloat16() for _ in range(2))
    logits = rnd(shared, h, sq, sk) * 3
    got = gpu_pkg.ops.batch_diffusion_cross_attention(q, m, logits, None, None, w_qg, w_kv, qb, h, out_dtype=torch.float32)
    heads = lambda x: x.bfloat16().double().view(batch, -1, h, c // h).transpose(1, 2).contiguous()
    (pq, pg), (pk, pv) = (x.double().matmul(w.double().t()).split(c, -1) for x, w in ((q, w_qg), (m, w_kv)))
    s = heads((pq + qb.double()) / (c // h) ** 0.5).matmul(heads(pk).transpose(2, 3).contiguous())
    s = s + logits.double()[torch.arange(batch, device="cuda") % shared]
    want = (s.softmax(-1).matmul(heads(pv)) * heads(torch.sigmoid(pg))).transpose(1, 2)
    scale = want.pow(2).mean().sqrt()
    assert (got - want).pow(2).mean().sqrt() <= 1e-2 * scale and (got - want).abs().max() <= 0.1 * scale
    # ... as if the entries that share it had been called by themselves
    for b in range(batch):
        one = gpu_pkg.ops.batch_diffusion_cross_attention(q[b:b + 1].contiguous(), m[b:b + 1].contiguous(), logits[b % shared][None].contiguous(),
                                                          None, None, w_qg, w_kv, qb, h, out_dtype=torch.float32)
        assert torch.equal(one[0], got[b])


@pytest.mark.gpu
@pytest.mark.parametrize("quads", [False, True])
@pytest.mark.parametrize("batch,n", [(1, 4), (2, 36), (1, 64), (2, 68), (5, 100), (1, 132), (1, 260)])
def test_what_lies_behind_the_last_key_is_not_read(gpu_pkg, batch, n, quads):
    """A last tile that is not full, and the tiles asked for past it, with NaN behind the projections and behind the logits: the bits
    of zeros in their place."""
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, h, lib = 768, 16, gpu_pkg.lib.load()
    x, w, qb = rnd(batch, n, c).bfloat16(), (rnd(4 * c, c) * 0.05).bfloat16(), rnd(c)
    plane = rnd(h, n, n) * 3
    if quads:
        plane = gpu_pkg.ops.quad_major_bias(plane)
    need, outs = lib.af3_batch_diffusion_self_attention_workspace_bytes(batch, n, c), []
    for behind in (0.0, float("nan")):
        ws = torch.full((need // 2 + 512 * 4 * c,), behind, dtype=torch.bfloat16, device="cuda")
        logits = torch.full((plane.numel() + 256 * (n + 4),), behind, device="cuda")
        logits[:plane.numel()] = plane.flatten()
        out = torch.empty(batch, n, h, c // h, device="cuda")
        gpu_pkg.lib.check(lib.af3_batch_diffusion_self_attention_forward(
            x.data_ptr(), None, 1, logits.data_ptr(), int(quads), w.data_ptr(), qb.data_ptr(), h, out.data_ptr(), gpu_pkg.lib.AF3_F32,
            batch, n, c, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream), "self-attention")
        outs.append(out)
    assert torch.isfinite(outs[1]).all() and torch.equal(*outs)
    assert torch.equal(outs[0], gpu_pkg.ops.batch_diffusion_self_attention(x, None, plane, w, qb, h, out_dtype=torch.float32))
