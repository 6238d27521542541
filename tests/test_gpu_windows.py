"""The windowed attention over gathered keys (four heads of 32 channels): the kernel that takes a whole window at once
against the general one on key tensors gathered beforehand, bit for bit, at the edges of its range: one query, a window
shorter than a tile of 64 keys, one just past it, one full; empty slots; padding masks; and the adaptive norm at every
number of 512-channel chunks."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sq,sk,windows,samples,masked", [
    (32, 128, 9, 5, True), (32, 128, 3, 1, False), (1, 4, 2, 2, False), (7, 60, 5, 2, True), (31, 64, 4, 3, True),
    (32, 68, 4, 1, True), (20, 124, 17, 2, False),
    (32, 128, 171, 3, True), (9, 60, 600, 1, True)])   # (the last two: more windows than two on every CU)
def test_windows_of_gathered_keys(gpu_pkg, sq, sk, windows, samples, masked):
    print(f"windows sq={sq} sk={sk} {windows}x{samples} masked={masked}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, atoms = 128, 50
    q, table = rnd(samples * windows, sq, c).bfloat16(), rnd(samples, atoms, c).bfloat16()
    rows = torch.randint(-3, atoms, (windows, sk), generator=g, device="cuda").clamp_min(-1).to(torch.int32)
    bias = rnd(windows, 4, sq, sk)
    mq = mk = None
    if masked:
        mq = (torch.rand(windows, sq, generator=g, device="cuda") > 0.3).float()
        mk = (torch.rand(windows, sk, generator=g, device="cuda") > 0.3).float()
    w = [(rnd(2 * c, c) * 0.1).bfloat16() for _ in range(2)]
    b = rnd(c)
    keys = table[:, rows.clamp_min(0).long()] * (rows >= 0)[None, ..., None]
    keys = keys.reshape(samples * windows, sk, c).bfloat16().contiguous()
    for dt in (torch.bfloat16, torch.float32):
        got = gpu_pkg.ops.gathered_cross_attention(q, table, rows, bias, mq, mk, w[0], w[1], b, 4, out_dtype=dt)
        want = gpu_pkg.ops.batch_diffusion_cross_attention(q, keys, bias, mq, mk, w[0], w[1], b, 4, out_dtype=dt)
        assert torch.isfinite(got).all() and torch.equal(got, want), float((got - want).abs().max())


@pytest.mark.parametrize("sq,sk", [(32, 128), (3, 8)])
def test_pair_logits_in_quads_of_keys(gpu_pkg, sq, sk):
    g = torch.Generator(device="cuda").manual_seed(sk)
    x, w = torch.randn(5, sq, sk, 16, generator=g, device="cuda"), torch.randn(12, 16, generator=g, device="cuda")
    ln = torch.rand(16, generator=g, device="cuda")
    rows = gpu_pkg.ops.atom_pair_logits(x, ln, w, 3, 4)
    quads = gpu_pkg.ops.atom_pair_logits(x, ln, w, 3, 4, quad_major=True)
    assert torch.equal(quads, rows.view(3, 5, 4, sq, sk // 4, 4).transpose(3, 4))


@pytest.mark.parametrize("rows,c,dtype", [(1, 16, torch.float32), (130, 128, torch.bfloat16), (16385, 128, torch.bfloat16), (37, 384, torch.bfloat16),
                                          (65, 768, torch.float32), (9, 1160, torch.bfloat16), (9, 2048, torch.float32)])
def test_adaptive_norm(gpu_pkg, rows, c, dtype):
    g = torch.Generator(device="cuda").manual_seed(rows + c)
    x = torch.randn(3 * rows, c, generator=g, device="cuda").to(dtype)
    ss = torch.randn(rows, 2 * c, generator=g, device="cuda")
    y = gpu_pkg.ops.layer_norm(x, scale=ss[:, :c], shift=ss[:, c:]).double()
    n = torch.nn.functional.layer_norm(x.double(), (c,))
    want = torch.sigmoid(ss[:, :c].double()).repeat(3, 1) * n + ss[:, c:].double().repeat(3, 1)
    assert ((y - want).abs() <= 1.01 * 2.0 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("n,dtype", [(1, torch.float32), (5, torch.bfloat16), (32, torch.float32), (67, torch.bfloat16), (132, torch.float32)])
def test_pair_logits_of_the_token_attention_in_quads(gpu_pkg, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(n)
    pair = torch.randn(n, n, 128, generator=g, device="cuda").to(dtype)
    w = torch.zeros(64, 128, device="cuda").bfloat16()
    w[:40] = torch.randn(40, 128, generator=g, device="cuda")
    ln = torch.rand(128, generator=g, device="cuda")
    rows = gpu_pkg.ops.pair_logits(pair, ln, None, w, 40)
    quads = gpu_pkg.ops.pair_logits(pair, ln, None, w, 40, quads=True)
    want = torch.nn.functional.pad(rows, (0, -n % 4)).view(40, n, -1, 4).transpose(1, 2)
    assert torch.equal(quads, want)


@pytest.mark.parametrize("sq,sk,windows", [(32, 128, 3), (7, 60, 5), (9, 60, 600)])
@pytest.mark.parametrize("poison", [float("nan"), float("inf")])
def test_an_empty_slot_reads_nothing(gpu_pkg, sq, sk, windows, poison):
    """Rows of the table that no slot names, row 0 and the last one among them, decide nothing."""
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    c, atoms = 128, 50
    q, table, bias = rnd(2 * windows, sq, c).bfloat16(), rnd(2, atoms, c).bfloat16(), rnd(windows, 4, sq, sk)
    rows = torch.randint(-8, atoms - 1, (windows, sk), generator=g, device="cuda")
    rows = torch.where(rows <= 0, torch.full_like(rows, -1), rows).to(torch.int32)
    w, b = [(rnd(2 * c, c) * 0.1).bfloat16() for _ in range(2)], rnd(c)
    run = lambda: gpu_pkg.ops.gathered_cross_attention(q, table, rows, bias, None, None, w[0], w[1], b, 4)
    want = run()
    table[:, 0] = table[:, -1] = poison
    assert torch.isfinite(want).all() and torch.equal(run(), want)
