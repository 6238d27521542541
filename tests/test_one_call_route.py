"""Where a run of modules goes to the library as one call: what that call is given, and which modules and arguments it
must not be made for.  Host side only (the operator layer is replaced by recorders); no GPU."""

import pytest
import torch


def test_outer_product_mean_epsilon_is_the_modules_at_the_call(pkg, monkeypatch):
    """Zero is a value like any other, and a change counts from the next call on, packed weights or not."""
    seen = []
    monkeypatch.setattr(pkg.ops, "outer_product_mean", lambda block, *a: seen.append(block.epsilon))
    monkeypatch.setattr(pkg.ops, "evoformer_stack", lambda blocks, *a: seen.extend(b.epsilon for b in blocks))
    blk = pkg.nn.EvoformerBlock()
    msa, pair = torch.zeros(2, 3, 64), torch.zeros(3, 3, 128)
    for eps in (1e-3, 0.0, 0.5):
        seen.clear()
        blk.outer_product_mean.epsilon = eps
        blk.outer_product_mean(msa, torch.ones(2, 3))
        blk(msa, pair, torch.ones(2, 3), torch.ones(3, 3))
        assert seen == [pytest.approx(eps)] * 2


def test_position_kernels_take_one_level(pkg):
    x, mask = torch.zeros(2, 3, 4, 3), torch.ones(3, 4)
    for levels in ((torch.ones(2, 1, 1, 1), None), (torch.ones(()), torch.ones(2))):
        with pytest.raises(ValueError, match="one element"):
            pkg.ops.positions(pkg.ops.POS_STEP, x, x, mask, *levels)
