"""Pairformer block (AF3 Algorithm 17, lines 2-8) and the trunk stack."""

from __future__ import annotations

import operator
from typing import Optional

import torch
import torch.nn as nn

from .. import check, ops
from .. import lib as L
from .attention import GridSelfAttention
from .base import (HipModule, as_written, bf16, drop_mesh, f32, fragments, in_check_mode, packs_of, pad_channels, pad_rows,
                   point)
from .diffusion_transformer import AdaLNZero, AdaptiveLayerNorm, SelfAttention
from .primitives import Transition
from .triangle_multiplication import TriangleMultiplication


def plain_pair_track(tm_out, tm_in, ta_start, ta_end, transition, c_pair) -> bool:
    """Whether the five pair operators are what one call of the library does: the triangle multiplications (outgoing,
    incoming), the triangle attentions (starting, ending node) and the transition, all on `c_pair` channels."""
    return (as_written((tm_out, TriangleMultiplication), (tm_in, TriangleMultiplication), (ta_start, GridSelfAttention),
                       (ta_end, GridSelfAttention), (transition, Transition))
            and c_pair == tm_out.c_pair == tm_in.c_pair == ta_start.c_pair == ta_end.c_pair == transition.c_x
            and tm_out._outgoing and not tm_in._outgoing and not ta_start.transpose and ta_end.transpose
            and ta_start.num_head == ta_end.num_head)


def one_sequence(single, seq_mask) -> bool:
    """Whether the single track is the one sequence that one call of the library knows ([N, c], mask [N]); a batch of
    them on one pair tensor runs module by module."""
    return single.dim() == 2 and (seq_mask is None or seq_mask.dim() == 1)


def fill_pair_weights(s, tm_out, tm_in, ta_start, ta_end, transition, c_pair, w_logits=None) -> torch.Tensor:
    """The pair operators' packed weights into an af3_pairformer_block; returns what only the structure points at."""
    vec, mat = (128,), (128, 128)
    for d, (tm, ta) in enumerate(((tm_out, ta_start), (tm_in, ta_end))):
        p, q = tm.packed(), ta.packed()
        point(s, (("tm_ln_in_w", d), p["ln_in_w"], vec), (("tm_ln_in_b", d), p["ln_in_b"], vec),
              (("tm_ln_c_w", d), p["ln_c_w"], vec), (("tm_ln_c_b", d), p["ln_c_b"], vec),
              (("tm_w_proj_gate", d), p["w_proj_gate"], (4, 128, 128)), (("tm_w_out", d), p["w_out"], mat),
              (("tm_w_gating", d), p["w_gl"], mat), (("ta_ln_w", d), q["ln_w"], vec), (("ta_ln_b", d), q["ln_b"], vec),
              (("ta_w_bias", d), q["w_bias"], (32, 128)), (("ta_w_qkvg", d), q["w_qkvg"], (4, 128, 128)),
              (("ta_w_out", d), q["w_out"], mat))
    p = transition.packed()
    hidden = p["w2"].shape[1]
    point(s, ("pt_ln_w", p["ln_w"], vec), ("pt_ln_b", p["ln_b"], vec), ("pt_w1", p["w1"], (hidden // 64, 128, 128)),
          ("pt_w2", p["w2"], (128, hidden)))
    s.valid_channels, s.num_head_pair, s.pair_hidden = c_pair, ta_start.num_head, hidden
    # (gathered first and reordered together: packing is paid for at every new set of weights)
    plain, turned, w2 = [], [], p["w2"]
    s.pair_channels = c = 64 if pair_of_64(ta_start, transition, c_pair) and w_logits is None else 128
    heads, d = ta_start.num_head, c_pair // ta_start.num_head
    for tm in (tm_out, tm_in):
        q = tm.packed()
        pg = q["w_proj_gate"]                        # 64 channels fill the first group of either operand
        plain += [q["w_gl"][:c, :c], q["w_out"][:c, :c], (pg if c == 128 else pg[::2, :, :c]).reshape(-1, c)]
    for ta in (ta_start, ta_end):
        q = ta.packed()
        qkvg, w_out = q["w_qkvg"], q["w_out"]
        if c == 64:                                  # without the padding of every head to 32 rows
            qkvg = qkvg.view(4, heads, 32, 128)[:, :, :d, :c].reshape(4, c, c)
            w_out = w_out.view(128, heads, 32)[:c, :, :d].reshape(c, c)
        plain += [qkvg[2], q["w_bias"][:, :c], w_out]
        turned += [qkvg[0:2].reshape(-1, c), qkvg[3]]
    plain.append(p["w1"][:, :, :c].reshape(-1, c))
    if w_logits is not None:
        plain.append(w_logits)
    frags = torch.cat([fragments(torch.cat(turned), swap23=True), fragments(torch.cat(plain)), fragments(w2[:c])])
    s.pair_frags = frags.data_ptr()
    return frags


def pair_of_64(att, transition, c_pair) -> bool:
    """Whether the library has kernels for the pair operators on 64 channels as they are (the template embedding of
    nn/d_template.py:198-201), without zero-padding the tensor to 128."""
    return c_pair == 64 and att.num_head == 4 and transition.packed()["w2"].shape[1] <= 128


def takes_64(s, pair: torch.Tensor) -> bool:
    """Whether a block whose structure is `s` takes this [N, N, 64] tensor as it is.  Its size decides and not its address:
    the statistics of a LayerNorm over zero-padded channels are rounded otherwise, and move outputs by bf16 places."""
    return s.pair_channels == 64 and pair.shape[0] <= L.PAIR64_MAX_TOKENS


def padded_128(s) -> "L.PairformerBlockStruct":
    """The structure for the same block on a tensor zero-padded to 128 channels."""
    if s.pair_channels != 64:
        return s
    p = L.PairformerBlockStruct.from_buffer_copy(s)
    p.device, p.pair_channels, p.pair_frags = s.device, 128, None
    return p


class PairformerBlock(HipModule):
    """Same constructor keywords, sub-module names and call signature as the
    reference's DistributePairformerBlock (nn/d_pairformer.py:32-106).

    As in the reference, `pair` and `single` are updated IN PLACE (`pair +=`,
    nn/d_pairformer.py:122-168) and returned; each of the seven sub-operations
    adds its update inside its last kernel instead of a separate pass."""

    def __init__(self, *args, n_heads: int = 16, c_pair: int = 128, c_single: int = 384,
                 c_hidden_mul: int = 128, n_heads_pair: int = 4, num_intermediate_factor: int = 4,
                 with_single: bool = True) -> None:
        super().__init__()
        args = drop_mesh(args)
        vals = list(args) + [n_heads, c_pair, c_single, c_hidden_mul, n_heads_pair, num_intermediate_factor,
                             with_single][len(args):]
        n_heads, c_pair, c_single, c_hidden_mul, n_heads_pair, num_intermediate_factor, with_single = vals[:7]
        self.n_heads, self.c_pair, self.c_single = n_heads, c_pair, c_single
        self.with_single, self.num_intermediate_factor = with_single, num_intermediate_factor
        self.triangle_multiplication_outgoing = TriangleMultiplication(c_pair=c_pair, _outgoing=True)
        self.triangle_multiplication_incoming = TriangleMultiplication(c_pair=c_pair, _outgoing=False)
        self.pair_attention1 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=False)
        self.pair_attention2 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=True)
        self.pair_transition = Transition(c_x=c_pair, num_intermediate_factor=num_intermediate_factor)
        if with_single:
            self.single_pair_logits_norm = nn.LayerNorm(c_pair)
            self.single_pair_logits_projection = nn.Linear(c_pair, n_heads, bias=False)
            self.single_attention_ = SelfAttention(c_x=c_single, num_head=n_heads, use_single_cond=False,
                                                   use_batch_infer=False)
            self.single_transition = Transition(c_x=c_single)

    def _pack(self):
        if not self.with_single:
            return {}
        return dict(ln_w=f32(self.single_pair_logits_norm.weight), ln_b=f32(self.single_pair_logits_norm.bias),
                    w_logits=pad_rows(bf16(self.single_pair_logits_projection.weight), 32))

    def _pair_track(self):
        m = self._modules
        return (m["triangle_multiplication_outgoing"], m["triangle_multiplication_incoming"], m["pair_attention1"],
                m["pair_attention2"], m["pair_transition"])

    @property
    def one_call(self) -> bool:
        """Whether the whole block runs as one call of the library (`native`): the fused pair operators, and a
        single track wide enough for the unfused transition."""
        track = self._pair_track()
        if not plain_pair_track(*track, self.c_pair):
            return False
        att = track[2]
        if not self.with_single:
            return att.fused or att.padded
        sa, st, c = self._modules["single_attention_"], self._modules["single_transition"], self.c_single
        if sa.__class__ is not SelfAttention:
            return False
        norm, out = sa._modules["adaptive_layernorm"], sa._modules["adaptive_zero_init"]
        return (att.fused and c > 128
                and as_written((sa, SelfAttention), (norm, AdaptiveLayerNorm), (out, AdaLNZero), (st, Transition))
                and c == sa.c_x == st.c_x and sa.num_head == self.n_heads and not norm.use_single_cond and not out.use_single_cond)

    def _structures(self):
        if self.one_call:
            self.native()

    def native(self) -> "L.PairformerBlockStruct":
        """The packed weights of the block's modules as the library's structure; made again when any of them has
        been packed again."""
        track = self._pair_track()
        mods = (self, *track)
        if self.with_single:
            sa, st = self._modules["single_attention_"], self._modules["single_transition"]
            mods += (sa, sa._modules["adaptive_layernorm"], sa._modules["adaptive_zero_init"], st)
        packs = packs_of(mods)
        if self._native is not None and all(map(operator.is_, self._native[1], packs)):
            return self._native[0]
        by = dict(zip(mods, packs))
        s = L.PairformerBlockStruct()
        frags = fill_pair_weights(s, *track, self.c_pair, by[self]["w_logits"] if self.with_single else None)
        s.with_single = int(self.with_single)
        if self.with_single:
            c, p, a, o, t = self.c_single, by[self], by[sa], by[sa.adaptive_zero_init], by[st]
            n, hidden = by[sa.adaptive_layernorm], t["w2"].shape[1]
            point(s, ("sl_ln_w", p["ln_w"], (128,)), ("sl_ln_b", p["ln_b"], (128,)),
                  ("sl_w", p["w_logits"], ((self.n_heads + 31) // 32 * 32, 128)),
                  ("sa_ln_w", n["ln_w"], (c,)), ("sa_ln_b", n["ln_b"], (c,)), ("sa_w_qkvg", a["w_qkvg"], (4 * c, c)),
                  ("sa_q_b", a["q_b"], (c,)), ("sa_w_out", o["w"], (c, c)), ("st_ln_w", t["ln_w"], (c,)),
                  ("st_ln_b", t["ln_b"], (c,)), ("st_w1", t["w1"], (2 * hidden, c)), ("st_w2", t["w2"], (c, hidden)))
            s.num_head, s.c_single, s.single_hidden = self.n_heads, c, hidden
        self._native = (s, packs, frags)
        return s

    def forward(self, pair: torch.Tensor, pair_mask: torch.Tensor, single: Optional[torch.Tensor] = None,
                seq_mask: Optional[torch.Tensor] = None, head: int = 0,
                single_stream: Optional["torch.cuda.Stream"] = None):
        """pair [N, N, c_pair], pair_mask [N, N], single [(B,) N, c_single], seq_mask [(B,) N].

        `single_stream` (not in the reference): run the update of `single` (attention and
        transition, a chain of small kernels that leave most of the GPU idle) on that
        stream, behind the pair-bias projection, and return without waiting for it.  The
        caller then owns the ordering: `single` may only be touched on that stream until
        the caller's stream has waited for it (PairformerStack does both)."""
        if in_check_mode():
            return check.pairformer_block(self, pair, pair_mask, single, seq_mask)
        if not pair.is_contiguous():
            raise ValueError("pair must be contiguous (it is updated in place)")
        if self.with_single and not single.is_contiguous():
            raise ValueError("single must be contiguous (it is updated in place)")
        if self.with_single and one_sequence(single, seq_mask) and self.one_call:
            ops.pairformer_stack([self.native()], pair, pair_mask, single, seq_mask, single_stream=single_stream,
                                 join=single_stream is None)
            return pair, single
        if not self.with_single and self.one_call:
            # (fewer than 128 channels and not the 64 that have kernels of their own: the five operators run on the
            # 128-channel kernels over one zero-padded copy of the tensor, which stays padded in between)
            s, x = self.native(), pair
            if self.c_pair < 128 and not takes_64(s, pair):
                s, x = padded_128(s), pad_channels(pair)
            elif self.c_pair < 128 and pair.data_ptr() % 16:     # the kernels' loads are of 16 bytes
                x = pair.clone()
            ops.pairformer_stack([s], x, pair_mask, None, None)
            if x is not pair:
                pair.copy_(x[..., :self.c_pair])
            return pair
        self.triangle_multiplication_outgoing.run(pair, pair_mask, residual=True)
        self.triangle_multiplication_incoming.run(pair, pair_mask, residual=True)
        self.pair_attention1.run(pair, pair_mask, residual=True)
        self.pair_attention2.run(pair, pair_mask, residual=True)
        self.pair_transition.run(pair, residual=True)
        if not self.with_single:
            return pair
        p = self.packed()
        # the only reader of `pair` on the single path: it stays on the caller's stream, in front of
        # whatever updates `pair` next
        logits = ops.pair_logits(pair, p["ln_w"], p["ln_b"], p["w_logits"], self.n_heads)
        if single_stream is None:
            self.single_attention_.run(single, seq_mask, logits, None, residual=True)
            self.single_transition.run(single, residual=True)
            return pair, single
        single_stream.wait_stream(torch.cuda.current_stream(pair.device))
        logits.record_stream(single_stream)
        with torch.cuda.stream(single_stream):
            self.single_attention_.run(single, seq_mask, logits, None, residual=True)
            self.single_transition.run(single, residual=True)
        return pair, single


_SIDE_STREAMS = {}


def _side_stream(device) -> "torch.cuda.Stream":
    """One extra stream per device (default priority), shared by every trunk loop of the process."""
    key = torch.device(device).index or 0
    if key not in _SIDE_STREAMS:
        _SIDE_STREAMS[key] = torch.cuda.Stream(device=device)
    return _SIDE_STREAMS[key]


def pairformer_loop(blocks, pair, pair_mask, single, seq_mask, overlap_single: bool = True):
    """Run Pairformer blocks one after the other (the loop of d_alphafold3.py:242-244).

    `overlap_single`: inside the loop nothing reads `single` but the next block's own
    single update, so each block's single update runs on a second stream while the next
    block's pair operators, which fill the GPU, run on the caller's; the caller's stream
    waits for the second one before the loop returns.  The results are the same bits
    either way."""
    if in_check_mode() or not overlap_single or not pair.is_cuda:
        for blk in blocks:
            pair, single = blk(pair, pair_mask, single, seq_mask)
        return pair, single
    side = _side_stream(pair.device)
    blocks = list(blocks)
    if blocks and one_sequence(single, seq_mask) and all(
            as_written((b, PairformerBlock)) and b.one_call and b.with_single and b.n_heads == blocks[0].n_heads
            and b.c_single == blocks[0].c_single for b in blocks):
        if not (pair.is_contiguous() and single.is_contiguous()):
            raise ValueError("pair and single must be contiguous (they are updated in place)")
        # (one block's update has nothing to run beside)
        ops.pairformer_stack([b.native() for b in blocks], pair, pair_mask, single, seq_mask,
                             single_stream=side if len(blocks) > 1 else None)
        return pair, single
    main = torch.cuda.current_stream(pair.device)
    side.wait_stream(main)          # whatever produced `single` and `seq_mask`
    for blk in blocks:
        pair, single = blk(pair, pair_mask, single, seq_mask, single_stream=side)
    main.wait_stream(side)
    return pair, single


class PairformerStack(HipModule):
    """The trunk loop of DistributeEvoformer.forward (d_alphafold3.py:242-244); see pairformer_loop."""

    def __init__(self, num_blocks: int = 48, overlap_single: bool = True, **block_kwargs) -> None:
        super().__init__()
        self.trunk_pairformer = nn.ModuleList([PairformerBlock(**block_kwargs) for _ in range(num_blocks)])
        self.overlap_single = overlap_single

    def _pack(self):
        return {}

    def forward(self, pair, pair_mask, single, seq_mask):
        return pairformer_loop(self.trunk_pairformer, pair, pair_mask, single, seq_mask, self.overlap_single)
