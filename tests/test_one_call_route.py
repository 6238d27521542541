"""Where a run of modules goes to the library as one call: what that call is given, and which modules and arguments it
must not be made for.  Host side only (the operator layer is replaced by recorders); no GPU."""

import copy
import ctypes
import gc
import inspect
import io
import re
import threading
import time
import weakref

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


def _small(nn, name):
    """A small module of each class that keeps the library's structures, and how it is brought to make them."""
    if name == "PairformerBlock":
        return nn.PairformerBlock(), lambda m: m.native()
    if name == "PairformerStack":
        return nn.PairformerStack(num_blocks=1), lambda m: m.trunk_pairformer[0].native()
    if name == "EvoformerBlock":
        return nn.EvoformerBlock(), lambda m: m.native()
    if name == "DiffusionTransformer":
        kw = dict(c_act=48, num_head=2, num_blocks=2, super_block_size=1)
        table = lambda m: nn.diffusion_transformer.block_table(m, list(zip(m.self_attention, m.transition_block)), 48)
        return nn.DiffusionTransformer(**kw), table
    table = lambda m: nn.diffusion_transformer.block_table(m, list(zip(m.cross_attention, m.transition_block)), 128)
    return nn.DiffusionCrossAttTransformer(num_blocks=1), table


NATIVE = ["PairformerBlock", "PairformerStack", "EvoformerBlock", "DiffusionTransformer", "DiffusionCrossAttTransformer"]


@pytest.mark.parametrize("name", NATIVE)
def test_packed_modules_can_be_copied_and_stored(pkg, name):
    mod, make = _small(pkg.nn, name)
    mod.load_hip_params()
    make(mod)
    stored = io.BytesIO()
    torch.save(mod, stored)
    stored.seek(0)
    for other in (copy.deepcopy(mod), torch.load(stored, weights_only=False)):      # (what this test has just written)
        assert all(torch.equal(a, b) for a, b in zip(mod.parameters(), other.parameters()))
        own, others = bytes(make(mod)), bytes(make(other))
        assert own != others          # the copy's structures point at weights of its own
    mod.__setstate__(dict(mod.__dict__, _packed={"of": "another version"}))
    assert mod._packed is None and mod._native is None


@pytest.mark.parametrize("name", NATIVE)
def test_invalidate_lets_go_of_the_packed_weights(pkg, name):
    mod, make = _small(pkg.nn, name)
    held = []
    make(mod)
    for m in mod.modules():
        if isinstance(m, pkg.nn.HipModule) and m._packed:
            held += [weakref.ref(t) for t in m._packed.values() if isinstance(t, torch.Tensor)]
    assert held
    params = {id(p) for p in mod.parameters()}
    mod.invalidate()
    gc.collect()
    assert all(r() is None or id(r()) in params for r in held)


def _hooked(m):
    m.register_forward_hook(lambda *a: None)


def _replaced(m):
    m.run = lambda *a, **k: None


def _another_class(m):
    m.__class__ = type("Derived", (type(m),), {})


@pytest.mark.parametrize("change", [_hooked, _replaced, _another_class])
def test_one_call_is_not_made_past_changed_modules(pkg, change):
    for cls, names in ((pkg.nn.PairformerBlock, ("pair_attention2", "triangle_multiplication_incoming", "pair_transition",
                                                 "single_transition", "single_attention_", "single_attention_.adaptive_layernorm")),
                       (pkg.nn.EvoformerBlock, ("outer_product_mean", "msa_attention1", "msa_transition", "pair_transition"))):
        assert cls().one_call
        for name in names:
            blk = cls()
            change(blk.get_submodule(name))
            assert not blk.one_call, name
    swapped = pkg.nn.PairformerBlock()
    swapped.pair_attention1.transpose = True
    assert not swapped.one_call


@pytest.mark.parametrize("change", [_hooked, _replaced, _another_class])
def test_transformers_are_not_run_past_changed_modules(pkg, change):
    dt = pkg.nn.diffusion_transformer

    def pairs(mod, att):
        return list(zip(getattr(mod, att), mod.transition_block))
    for make, att, cls, norms, heads in (
            (lambda: dt.DiffusionTransformer(c_act=48, num_head=2, num_blocks=2, super_block_size=1), "self_attention",
             dt.SelfAttention, ("adaptive_layernorm",), 2),
            (lambda: dt.DiffusionCrossAttTransformer(num_blocks=2), "cross_attention", dt.CrossAttention,
             ("q_adaptive_layernorm", "k_adaptive_layernorm"), 4)):
        assert dt.plain_blocks(pairs(make(), att), norms, cls, heads)
        for name in [f"{att}.1", "transition_block.1", "transition_block.0.adaptive_zero_init"] + [f"{att}.0.{k}" for k in norms]:
            mod = make()
            change(mod.get_submodule(name))
            assert not dt.plain_blocks(pairs(mod, att), norms, cls, heads), name


def test_scratch_is_checked_for_every_block_before_anything_is_launched(pkg):
    lib, some = pkg.lib.load(), 1 << 20      # (an address that is not null: nothing is to touch it)
    n, narrow, wide = 16, pkg.lib.PairformerBlockStruct(), pkg.lib.PairformerBlockStruct()
    for b, hidden in ((narrow, 1536), (wide, 3456)):
        b.valid_channels, b.num_head_pair, b.with_single, b.num_head, b.c_single, b.single_hidden = 128, 4, 1, 16, 384, hidden
    pair_ws = lib.af3_pairformer_stack_workspace_bytes(n, 4)
    need = lib.af3_pairformer_single_workspace_bytes(n, 384, 1536)
    assert need < lib.af3_pairformer_single_workspace_bytes(n, 384, 3456)

    def call(blocks, wsb, swsb):
        ptrs = (ctypes.c_void_p * len(blocks))(*[ctypes.addressof(b) for b in blocks])
        return lib.af3_pairformer_stack_forward(ptrs, len(blocks), some, 0, None, None, some, 0, None, n, some, some, wsb, some,
                                                swsb, None, None, 1)
    assert call([narrow, wide], pair_ws, need) == -2
    assert call([narrow], pair_ws, need - 1) == -2 and call([narrow], pair_ws - 1, need) == -2
    wide.c_single = 256
    assert call([narrow, wide], pair_ws, 1 << 30) == -1

    m = pkg.lib.MsaBlockStruct()
    m.pair.num_head_pair = 4
    ptrs = (ctypes.c_void_p * 1)(ctypes.addressof(m))
    msa_ws = lib.af3_msa_workspace_bytes(8, n)
    for a, b in ((msa_ws - 1, pair_ws), (msa_ws, pair_ws - 1)):
        assert lib.af3_evoformer_stack_forward(ptrs, 1, some, 0, some, some, 0, None, 8, n, some, a, some, b, None) == -2


class _General(Exception):
    """The general kernels were called."""


@pytest.mark.parametrize("rows,n,mask_rows,taken", [(2, 8192, 2, True), (2, 8193, 2, False), ((1 << 24) + 1, 64, (1 << 24) + 1, False),
                                                    (4, 6, 1, False)])
def test_msa_sizes_and_masks_beyond_the_msa_kernels_go_to_the_general_ones(pkg, monkeypatch, rows, n, mask_rows, taken):
    opm, att, blk = pkg.nn.OuterProductMean(), pkg.nn.MSAAttention(), pkg.nn.EvoformerBlock()
    for m in (opm.packed, att.packed, blk.native):
        m()
    zero = torch.zeros(1)                    # (tensors without memory of their own, and nothing that would give them any)
    msa, pair, mask = zero.expand(rows, n, 64), zero.expand(n, n, 128), zero.expand(mask_rows, n)
    for name in ("contiguous", "float"):
        monkeypatch.setattr(torch.Tensor, name, lambda t: t)
    monkeypatch.setattr(torch.Tensor, "is_contiguous", lambda t: True)

    def general(*a, **k):
        raise _General
    monkeypatch.setattr(pkg.ops, "layer_norm", general)
    for name in ("outer_product_mean", "msa_attention", "evoformer_stack"):
        monkeypatch.setattr(pkg.ops, name, lambda *a, **k: "own")
    for call in (lambda: opm.run(msa, mask, residual=pair), lambda: att.run(msa, mask, pair, True),
                 lambda: blk(msa, pair, mask, zero.expand(n, n))):
        if taken:
            call()
        else:
            with pytest.raises(_General):
                call()


def test_a_strided_tensor_goes_to_the_padded_transition(pkg, monkeypatch):
    monkeypatch.setattr(pkg.ops, "transition128", lambda x, *a, **k: x + 1)
    x = torch.zeros(64, 6).t()
    assert pkg.nn.Transition(c_x=64).run(x, True) is x and bool((x == 1).all())


@pytest.mark.parametrize("name,layer,widths", [
    ("PairformerBlock", "pair_transition.transition2", (256, 128)),
    ("PairformerBlock", "single_attention_.adaptive_zero_init.transition2", (256, 384)),
    ("PairformerBlock", "pair_attention1.output_projection", (64, 128)),
    ("EvoformerBlock", "msa_attention1.gating_query", (32, 64)),
    ("EvoformerBlock", "msa_transition.transition1", (64, 128)),
    ("DiffusionTransformer", "self_attention.1.adaptive_zero_init.transition2", (24, 48)),
    ("DiffusionCrossAttTransformer", "transition_block.0.transition1", (128, 256))])
def test_weights_of_another_shape_are_refused(pkg, name, layer, widths):
    """The structures carry addresses without sizes: a kernel would read past a smaller weight."""
    mod, make = _small(pkg.nn, name)
    parent, _, leaf = layer.rpartition(".")
    setattr(mod.get_submodule(parent), leaf, torch.nn.Linear(*widths, bias=False))
    mod.load_hip_params()                    # (packing is no use of the weights)
    with pytest.raises(ValueError, match="expected a weight"):
        make(mod)


def test_packed_weights_are_contiguous_and_of_the_librarys_types(pkg):
    """What the structures take for granted of every address."""
    nn = pkg.nn
    for mod in (nn.PairformerBlock(), nn.PairformerBlock(c_pair=64, num_intermediate_factor=2, with_single=False),
                nn.EvoformerBlock(), nn.DiffusionTransformer(c_act=48, num_head=2, num_blocks=1, super_block_size=1),
                nn.DiffusionCrossAttTransformer(num_blocks=1)):
        mod.half()                               # (whatever the parameters are)
        mod.load_hip_params()
        for m in mod.modules():
            for k, t in (getattr(m, "_packed", None) or {}).items():
                for t in t if isinstance(t, list) else [t]:
                    want = torch.float32 if t.dim() == 1 or k == "w_f32" else torch.bfloat16
                    assert t.dtype == want and t.is_contiguous(), (type(m).__name__, k, t.dtype)


def test_weights_on_another_device_are_refused(pkg):
    """The addresses of weights that are still on the CPU are nothing a kernel may be given."""
    nn, ops = pkg.nn, pkg.ops
    for name in NATIVE:
        mod, make = _small(nn, name)
        native = make(mod)
        assert native.device == torch.device("cpu")
        with pytest.raises(ValueError, match="weights: live on cpu"):
            ops._weights_with(torch.empty(1, device="meta"), native)
        ops._weights_with(torch.empty(1), native)
    blk = nn.EvoformerBlock()
    blk.pair_transition._packed = {k: v.to("meta") for k, v in blk.pair_transition.packed().items()}
    with pytest.raises(ValueError, match="other weights of the block on cpu"):
        blk.native()


def test_an_index_tensor_that_was_written_to_is_checked_again(pkg):
    """The kernels read the rows that an index tensor names; a check of earlier contents is none of the present ones."""
    rows = torch.tensor([0, 3, -1], dtype=torch.int32)
    for _ in range(2):
        pkg.ops.rows_in_range(rows, 4)
    rows[2] = 4
    with pytest.raises(ValueError, match="beyond"):
        pkg.ops.rows_in_range(rows, 4)
    pkg.ops.rows_in_range(rows, 5)
    with pytest.raises(ValueError, match="beyond"):
        pkg.ops.rows_in_range(rows, 4)
    with torch.inference_mode():
        pkg.ops.rows_in_range(rows.clone(), 5)


def test_foreign_modules_are_not_taken_for_the_usual_ones(pkg):
    nn, foreign = pkg.nn, torch.nn.Identity
    blk = nn.PairformerBlock()
    for name in ("pair_attention1", "single_attention_", "single_transition", "pair_transition"):
        other = nn.PairformerBlock()
        setattr(other, name, foreign())
        assert blk.one_call and not other.one_call
    mod = nn.DiffusionTransformer(c_act=48, num_head=2, num_blocks=2, super_block_size=1)
    assert mod._one_call(mod._blocks())
    mod.transition_block[1] = foreign()
    assert not mod._one_call(mod._blocks())


@pytest.mark.parametrize("name", NATIVE)
def test_packing_makes_the_structures_too(pkg, name):
    mod, make = _small(pkg.nn, name)
    mod.load_hip_params()
    holder = mod.trunk_pairformer[0] if name == "PairformerStack" else mod
    held = holder._native
    assert held is not None and make(mod) is held[0]


def test_operators_with_scratch_run_one_at_a_time(pkg):
    """Two threads on one stream share its scratch."""
    inside, worst = [], []

    @pkg.ops._uses_scratch
    def op():
        inside.append(1)
        worst.append(len(inside))
        time.sleep(0.002)
        inside.pop()
    threads = [threading.Thread(target=lambda: [op() for _ in range(10)]) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(worst) == 40 and max(worst) == 1
    source = inspect.getsource(pkg.ops)
    users = re.findall(r"^(@_uses_scratch\n)?def (\w+)\((?:(?!^def ).)*? = _ws\(", source, flags=re.M | re.S)
    assert len(users) >= 11 and all(mark for mark, name in users), users
