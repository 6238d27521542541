"""The element-wise passes of the trunk's embedding and of the diffusion head against the torch operations they stand for,
bit for bit: clipped offsets of every kind, bonds with a masked end and at [0, 0], one atom and odd counts."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 150])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_trunk_pair_embedding(gpu_pkg, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    batch = gpu_pkg.nn.atom_layout.synthetic_trunk_batch(n, 2, torch.Generator().manual_seed(n), chain_len=61).to("cuda")
    tok, trunk = batch.token_features, gpu_pkg.nn.trunk.Evoformer
    tok.token_index = (torch.arange(n, device="cuda") * 7) % (n + 1)          # offsets within a residue, clipped and not
    tok.residue_index = torch.div(torch.arange(n, device="cuda"), 2, rounding_mode="floor")
    lr, prev, wpos, bond = rnd(n, 300), rnd(n, n, 128), rnd(139, 128), rnd(128)
    rel = gpu_pkg.nn.diffusion_head.create_relative_encoding(tok, 32, 2)
    contact = trunk.contact_matrix(batch, n, "cuda")
    want = lr[:, None, :128] + lr[None, :, 128:256] + prev
    want = want + wpos[rel[..., :66].argmax(-1)] + wpos[66 + rel[..., 66:132].argmax(-1)]
    want = want + rel[..., 132:133].float() * wpos[132] + wpos[133 + rel[..., 133:].argmax(-1)]
    want = (want + contact[:, :, None] * bond).to(dtype)
    got_c = gpu_pkg.ops.contact_matrix((batch.polymer_ligand_bond_info.tokens_to_polymer_ligand_bonds,
                                        batch.ligand_ligand_bond_info.tokens_to_ligand_ligand_bonds), n, "cuda")
    assert torch.equal(got_c, contact)
    ids = [getattr(tok, k).long() for k in ("asym_id", "residue_index", "token_index", "entity_id", "sym_id")]
    assert torch.equal(gpu_pkg.ops.pair_embed(lr, prev, ids, wpos, bond, got_c, dtype), want)
    a = rnd(3, n, 64)
    assert torch.equal(gpu_pkg.ops.add_rows(a, lr[:, 256 - 64:256], dtype), (a + lr[:, 192:256]).to(dtype))
    x, m = a.bfloat16(), torch.rand(n, generator=g, device="cuda")
    assert torch.equal(gpu_pkg.ops.mask_rows(x.clone(), m), x * m.bfloat16()[:, None])


@pytest.mark.parametrize("samples,n,atoms", [(1, 1, 1), (5, 33, 24)])
def test_position_passes(gpu_pkg, samples, n, atoms):
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y, mask = rnd(samples, n, atoms, 3), rnd(samples, n, atoms, 3), (rnd(n, atoms) > 0).float()
    levels, am, ops = torch.rand(3, generator=g, device="cuda") * 50, mask[None, ..., None], gpu_pkg.ops
    t, nx = levels[0], levels[1]
    root = torch.sqrt(t ** 2 + 16.0 ** 2)
    assert torch.equal(ops.positions(ops.POS_SCALE, x, None, mask, t), x * am / root)
    blend = (16.0 ** 2 / (t ** 2 + 16.0 ** 2) * x + t * 16.0 / root * y) * am
    assert torch.equal(ops.positions(ops.POS_BLEND, x, y, mask, t), blend)
    shift = rnd(3)
    assert torch.equal(ops.positions(ops.POS_PLACE, x, shift, mask, t), (x + shift) * am + t)
    step = x + 1.5 * (nx - t) * ((x - y) / t)
    assert torch.equal(ops.positions(ops.POS_STEP, x, y, None, t, nx, 1.5), step)
