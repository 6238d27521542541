"""GPU parity of the dense products below the 256x256-tile sizes, one case at the edges of every tile the launcher
chooses from (32x32, 64x64, 64x128, 128x128, the element-wise form), and of the large tile: first and last rows and columns alone in a tile,
K shorter than a slab, K with a partial last slab, column counts that force element-wise stores; the order of
summation, which must not depend on the number of rows; and the K split of the Pairformer's single track."""

import pytest
import torch

from oracle import af3_oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 8, 8), (33, 40, 320), (64, 384, 384), (97, 72, 1536), (500, 768, 128),        # 32x32
    (387, 1536, 384), (65, 8200, 64), (12001, 64, 64), (1921, 768, 768),              # 64x64, four and three buffers
    (3841, 768, 768), (129, 12352, 384), (70001, 64, 320),                            # 64x64, two buffers
    (12001, 136, 120), (129, 3072, 392), (97, 72, 1032),                              # 64x64, K with a partial last slab
    (31, 3, 64), (97, 65, 200), (500, 765, 392),                                      # 64x64, element by element
    (1921, 3080, 128), (8001, 384, 1024), (70, 70016, 64), (180001, 128, 64),         # 64x128
    (8000, 1024, 104), (7777, 2112, 40), (30720, 256, 192),                           # 256x256: K in one, two, three slabs
    (1249, 3072, 512), (1985, 3072, 512), (2113, 3072, 64), (8961, 768, 128), (4225, 768, 1024),   # 128x128, 128x192, eight waves
    (513, 3008, 128), (513, 3008, 384), (571, 3072, 384),     # SwiGLU in 64x64 and 128x64
    (2753, 768, 384), (2688, 768, 384), (699, 3072, 384),     # 64x64, just past and below two tiles to a CU
    (20001, 1032, 128),                      # 128x128 (odd columns keep it off the large tile)
]


def ulp_ok(name, got, want, atol=2e-4):
    got, want = got.double().cpu(), want.double().cpu()
    bad = (got - want).abs() > 1.01 * 2.0 ** -8 * want.abs() + atol
    assert not bad.any(), f"{name}: {int(bad.sum())} elements beyond one bf16 ulp"


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_epilogues(gpu_pkg, m, n, k):
    print(f"dense tiles m={m} n={n} k={k}", flush=True)
    ops, L = gpu_pkg.ops, gpu_pkg.lib
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, w, b = rnd(m, k).bfloat16(), (rnd(n, k) * 0.1).bfloat16(), rnd(n)
    y = x.float() @ w.float().t()
    ulp_ok("fp32, bias, scale", ops.linear(x, w, bias=b, alpha=0.5, out_dtype=torch.float32), (y + b) * 0.5)
    ulp_ok("sigmoid", ops.linear(x, w, bias=b, sigmoid=True), torch.sigmoid(y + b))
    gate = torch.rand(1 if m % 7 else 7, n, generator=g, device="cuda")
    rows = gate.repeat(m // gate.shape[0], 1)
    for dt in (torch.bfloat16, torch.float32):
        res = rnd(m, n).to(dt)
        want = y * rows + res.float()
        out = ops.linear(x, w, out_dtype=dt, mode=L.LINEAR_GATE_RES, gate=gate, residual=res, out=res)
        assert out is res
        ulp_ok(f"gate, residual in place {dt}", out, want)
    if n % 64 == 0:
        h = ops.linear(x, w, mode=L.LINEAR_SWIGLU)
        a, c = y.view(m, n // 64, 2, 32).unbind(2)
        ulp_ok("swiglu", h, (torch.nn.functional.silu(a) * c).reshape(m, n // 2))
    if m % 32 == 0 and n % 32 == 0:
        r = ops.linear(x, w, mode=L.LINEAR_REGROUP32)
        ulp_ok("regrouped", r, y.view(m // 32, 32, n // 32, 32).transpose(1, 2).reshape(-1, 1024))


@pytest.mark.parametrize("batch,m,n,k", [(128, 64, 64, 64), (128, 61, 61, 64), (3, 130, 24, 72), (8, 100, 300, 104)])
def test_batched_product(gpu_pkg, batch, m, n, k):
    print(f"dense tiles batch={batch} m={m} n={n} k={k}", flush=True)
    g = torch.Generator().manual_seed(m)
    a, b = (O.round_bf16(torch.randn(batch, s, k, generator=g)) for s in (m, n))
    got = gpu_pkg.ops.batched_nt_product(a.cuda().bfloat16(), b.cuda().bfloat16())
    ulp_ok("batched", got, torch.stack([p.double() @ q.double().t() for p, q in zip(a, b)]))


@pytest.mark.parametrize("n,k", [(768, 768), (384, 1536), (128, 128), (3072, 768)])
def test_rows_do_not_change_with_the_batch(gpu_pkg, n, k):
    """Every tile sums K in the same order, so the first rows of a product are the same bits however many follow."""
    print(f"dense tiles: batch invariance n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(9000, k, generator=g, device="cuda").bfloat16()
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.1).bfloat16()
    want = gpu_pkg.ops.linear(x, w, mode=gpu_pkg.lib.LINEAR_GATE_RES)
    for m in (1, 100, 500, 1900, 3840):
        assert torch.equal(gpu_pkg.ops.linear(x[:m], w, mode=gpu_pkg.lib.LINEAR_GATE_RES), want[:m]), m


@pytest.mark.parametrize("n,c", [(1, 384), (33, 384), (130, 384), (700, 384), (1000, 256)])
def test_single_track_products(gpu_pkg, n, c):
    """The single track of a Pairformer block, whose products may split K between waves (by four, eight and two),
    against the same modules run one by one, whose products do not."""
    print(f"dense tiles: single track n={n} c={c}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + c)
    with torch.device("cuda"):
        blk = gpu_pkg.nn.PairformerBlock(c_single=c, n_heads=c // 32)
    with torch.no_grad():
        for p in blk.parameters():
            p.normal_(0.0, 0.05, generator=g)
    blk.invalidate()
    pair = torch.randn(n, n, 128, generator=g, device="cuda").bfloat16()
    single = torch.randn(n, c, generator=g, device="cuda")
    mask = torch.ones(n, device="cuda")
    ones = torch.ones(n, n, device="cuda")
    out_pair, got = blk(pair.clone(), ones, single.clone(), mask)
    p = blk.packed()
    logits = gpu_pkg.ops.pair_logits(out_pair, p["ln_w"], p["ln_b"], p["w_logits"], blk.n_heads)
    want = single.clone()
    blk.single_attention_.run(want, mask, logits, None, residual=True)
    blk.single_transition.run(want, residual=True)
    upd, ref = got - single, want - single
    assert float((upd - ref).norm() / ref.norm()) < 3e-3
