"""The start of a sampling step in one kernel (augment_positions_kernel)."""

import pytest
import torch


# one atom; the last a workgroup keeps in registers and the first it does not; no atom at all under the mask
@pytest.mark.gpu
@pytest.mark.parametrize("samples,n,atoms,masked", [(1, 1, 1, 0.0), (5, 33, 24, 0.5), (2, 1024, 8, 0.1), (3, 8193, 1, 0.1), (2, 1003, 24, 0.4),
                                                    (2, 7, 24, 1.0)])
def test_against_64_bits(gpu_pkg, samples, n, atoms, masked):
    """Each sum of up to 24072 atoms in runs of at most 24 and trees of 64 and 16: 30 roundings of its terms' size on the centre, and
    a dozen on the way to the result."""
    g = torch.Generator(device="cuda").manual_seed(n + atoms)
    x = torch.randn(samples, n, atoms, 3, generator=g, device="cuda") * 50 + 20
    mask = (torch.rand(n, atoms, generator=g, device="cuda") >= masked).float()
    rot = gpu_pkg.nn.diffusion_head.random_rotation(g, "cuda")
    shift, noise = torch.randn(3, generator=g, device="cuda"), torch.rand(4, generator=g, device="cuda")[2]
    got = gpu_pkg.ops.augment_positions(x, rot, shift, mask, noise)
    want = gpu_pkg.nn.diffusion_head.random_augmentation(x.double(), mask[None], rot.double(), shift.double()) + noise.double()
    assert (got.double() - want).abs().max() <= 48 * 2.0 ** -24 * (x.abs().max() * 2 + 4)
    assert torch.equal(got[:, mask == 0], noise.expand_as(got[:, mask == 0]))


def test_refused(pkg):
    lib = pkg.lib.load()
    one, two = 1 << 20, 1 << 21
    assert lib.af3_augment_positions_forward(one, one, one, one, one, one, 1, 8, None) == -1     # in place
    assert lib.af3_augment_positions_forward(one, None, one, one, one, two, 1, 8, None) == -1
    assert lib.af3_augment_positions_forward(one, one, one, one, one, two, 1, 0, None) == -1
