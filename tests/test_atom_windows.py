"""The windows of the atom cross-attention that nobody reads are left out (embed.hip, atom_windows_kernel; atom_step.hip; attention.hip,
window_kernel)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _list(pkg, mask, idx, exists, keys):
    out = pkg.ops.atom_windows(mask, idx, exists, keys).cpu()
    return out[1:1 + int(out[0])].tolist()


@pytest.mark.parametrize("s,q", [(1, 32), (5, 32), (33, 4), (1023, 32), (1025, 32), (2500, 7)])
def test_the_windows_that_are_read(gpu_pkg, s, q):
    """Against the definition; a key that leads to a row which nothing names asks for all."""
    g = torch.Generator().manual_seed(s)
    mask = (torch.rand(s, q, generator=g) < 0.02).float() * (torch.arange(s) % 3 != 0)[:, None]
    idx = torch.randint(0, s * q, (s, 9), generator=g)
    exists = torch.rand(s, 9, generator=g) < 0.05
    want = (mask != 0).reshape(-1)
    want[idx[exists]] = True
    keys = torch.where(torch.rand(s, 16, generator=g) < 0.5, torch.randint(0, s * q, (s, 16), generator=g), -1)
    keys = torch.where((keys >= 0) & want[keys.clamp(min=0)], keys, -1).to(torch.int32)
    dev = lambda *t: [x.cuda().contiguous() for x in t]
    expect = want.reshape(s, q).any(-1).nonzero().flatten().tolist()
    assert _list(gpu_pkg, *dev(mask, idx, exists, keys)) == expect
    if not want.all():
        keys[-1, -1] = int((~want).nonzero()[-1])
        assert _list(gpu_pkg, *dev(mask, idx, exists, keys)) == list(range(s))
    nothing = torch.zeros_like(exists)
    assert _list(gpu_pkg, *dev(torch.zeros_like(mask), idx, nothing, torch.full_like(keys, -1))) == []
    assert _list(gpu_pkg, *dev(torch.ones_like(mask), idx, nothing, keys)) == list(range(s))


@pytest.mark.parametrize("n,padding,samples", [(8, 0, 1), (20, 3, 5), (64, 40, 2), (104, 9, 3)])
def test_positions_are_those_of_all_windows(gpu_pkg, monkeypatch, n, padding, samples):
    """The same bits, at the first evaluation on a state and at the next; and from a layout in which some atoms' windows are read only
    on the way back."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    with torch.device("cuda"):
        head = gpu_pkg.nn.DiffusionHead(num_blocks=1)
    with torch.no_grad():
        for name, p in head.named_parameters():
            p.normal_(0.0, 0.05, generator=gen)
            if p.dim() == 1 and name.endswith("weight"):
                p += 1.0
    head.invalidate()
    batch = gpu_pkg.nn.atom_layout.synthetic_batch(n, torch.Generator().manual_seed(n), n_padding_tokens=padding).to("cuda")
    emb = {"single": rnd(n, 384), "pair": rnd(n, n, 128), "target_feat": rnd(n, 447)}
    level = torch.tensor([3.0], device="cuda")
    pos = [rnd(samples, n, 24, 3) for _ in range(2)]
    single, pair = head.pre_conditioning(batch, emb, level, True)

    def run():
        state = head.prepare(batch, emb, pair)
        return state, [head(x, level[0], batch, emb, single[0], pair, state=state) for x in pos]
    state, got = run()
    live = int(state.encoder.windows[0])
    assert 0 < live < state.encoder.windows.numel() - 1
    monkeypatch.setattr(gpu_pkg.ops, "atom_windows", lambda *a: None)
    state, want = run()
    assert state.encoder.windows is None
    for x, y in zip(got, want):
        assert torch.isfinite(x).all() and x.abs().max() > 0 and torch.equal(x, y)
