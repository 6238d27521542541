"""Evoformer (MSA) block: outer-product mean, MSA pair-weighted averaging, MSA
transition and the five pair operators (nn/d_pairformer.py:174-252,
nn/d_primitives.py:42-70, nn/d_attention.py:113-156).  Same constructor
keywords, parameter names and `forward` signatures as the reference's
Distribute* classes; msa and pair are updated in place as the reference's `+=`.

Both MSA operators are products over long axes and run on the bf16 MFMA
kernels; at the width of the published model (64 channels) a run of blocks is one
call of the library (`evoformer_loop`).
  * outer-product mean: out[b, d, :] = W^T vec(sum_a L[a, b, :] (x) R[a, d, :]).
    The sum over the MSA rows is one product [(b, c), a] x [(d, e), a]^T whose
    tiles, 8 x 8 token pairs' outer products, are multiplied with W where they
    arise: neither the [N, N, 32, 32] tensor that the reference's einsum
    materialises (1.2 GB) nor any part of it goes to memory.
  * pair-weighted averaging: per head, softmax(pair logits) [q, k] times the
    head's values of all MSA rows [(row, channel), k]^T.
Both sum over an index (MSA rows, tokens) that the activations [rows, N, c]
carry as an outer one, while the dense kernels want it innermost: the
projections are written transposed.  Other widths go operator by operator
through the general kernels; there the operands are produced transposed
(projection weights as the left operand) or run through the bf16 transpose
kernel where rows and tokens are multiples of 8, and through strided copies
elsewhere.
"""

from __future__ import annotations

import operator
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import check, ops
from .. import lib as L
from .attention import GridSelfAttention
from .base import HipModule, as_written, bf16, drop_mesh, f32, in_check_mode, packs_of, pad_rows, point
from .pairformer import fill_pair_weights, plain_pair_track
from .primitives import Transition
from .triangle_multiplication import TriangleMultiplication


def _pad_last(x: torch.Tensor, multiple: int = 8) -> torch.Tensor:
    k = x.shape[-1]
    return x if k % multiple == 0 else F.pad(x, (0, (-k) % multiple))


def _takes(msa, mask) -> bool:
    """Whether the MSA track's own kernels take these: their range of sizes, and one mask value per position (the general
    kernels also take masks that broadcast)."""
    return ops.msa_in_range(*msa.shape[:2]) and mask.shape == msa.shape[:2]


class OuterProductMean(HipModule):
    """nn/d_primitives.py:42-70."""

    def __init__(self, *args, c_msa: int = 64, num_output_channel: int = 128, num_outer_channel: int = 32,
                 epsilon: float = 1e-3) -> None:
        super().__init__()
        args = drop_mesh(args)
        vals = list(args) + [c_msa, num_output_channel, num_outer_channel][len(args):]
        c_msa, num_output_channel, num_outer_channel = vals[:3]
        self.c_msa, self.num_output_channel, self.num_outer_channel = c_msa, num_output_channel, num_outer_channel
        self.epsilon = epsilon
        self.layer_norm_input = nn.LayerNorm(c_msa)
        self.left_projection = nn.Linear(c_msa, num_outer_channel, bias=False)
        self.right_projection = nn.Linear(c_msa, num_outer_channel, bias=False)
        self.output_w = nn.Parameter(torch.zeros(num_outer_channel, num_outer_channel, num_output_channel))
        self.output_b = nn.Parameter(torch.zeros(num_output_channel))

    @property
    def native(self) -> bool:
        return self.c_msa == 64 and self.num_outer_channel == 32 and self.num_output_channel == 128

    def _pack(self):
        co = self.num_outer_channel
        d = dict(ln_w=f32(self.layer_norm_input.weight), ln_b=f32(self.layer_norm_input.bias),
                    w_l=bf16(self.left_projection.weight), w_r=bf16(self.right_projection.weight),
                    w_out=bf16(self.output_w.detach().reshape(co * co, -1).t()), b_out=f32(self.output_b))
        if self.native:
            d["w_lr"] = torch.cat([d["w_l"], d["w_r"]])
            rows = [(r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1) for r in range(32)]
            d["w_packed"] = d["w_out"].view(4, 32, 64, 2, 8)[:, rows].permute(0, 2, 3, 1, 4).contiguous()
        return d

    def block(self) -> "L.MsaBlockStruct":
        """The packed weights as the library's structure, epsilon as it is now (an attribute, not a weight)."""
        d = self.packed()
        if self._native is None or self._native[1] is not d:
            s = L.MsaBlockStruct()
            point(s, ("opm_ln_w", d["ln_w"], (64,)), ("opm_ln_b", d["ln_b"], (64,)), ("opm_w_lr", d["w_lr"], (64, 64)),
                  ("opm_w_out", d["w_packed"], (4, 64, 2, 32, 8)), ("opm_b_out", d["b_out"], (128,)))
            self._native = (s, d)
        self._native[0].epsilon = self.epsilon
        return self._native[0]

    def _structures(self):
        if self.native:
            self.block()

    @torch.no_grad()
    def run(self, msa, mask, residual: Optional[torch.Tensor] = None, block: int = 128):
        """-> [N, N, c_pair] fp32, or `residual` (the pair tensor) updated in place."""
        p = self.packed()
        a, n, _ = msa.shape
        co, cf = self.num_outer_channel, self.num_output_channel
        out = residual if residual is not None else torch.zeros((n, n, cf), dtype=torch.float32, device=msa.device)
        if self.native and _takes(msa, mask):
            return ops.outer_product_mean(self.block(), msa.contiguous(), mask, out, True)
        m = mask.float()
        x = ops.layer_norm(msa.contiguous(), p["ln_w"], p["ln_b"])
        mb = m[..., None].to(torch.bfloat16)

        def projected(w):        # [(token, channel), MSA row]: the summation index innermost
            y = ops.linear(x, w) * mb                                                       # [a, N, co]
            if a % 8 == 0 and (n * co) % 8 == 0:
                return ops.transpose2d(y.view(a, n * co))
            return _pad_last(y.permute(1, 2, 0).reshape(n * co, a)).contiguous()
        lt, rt = projected(p["w_l"]), projected(p["w_r"])
        inv_norm = (1.0 / (self.epsilon + m.t() @ m)).contiguous()                         # [b, d]
        for b0 in range(0, n, block):
            b1 = min(n, b0 + block)
            if co == 32:
                outer = ops.linear(lt[b0 * co:b1 * co], rt, mode=ops._L.LINEAR_REGROUP32)  # [(b, d), (c, e)]
            else:
                outer = ops.linear(lt[b0 * co:b1 * co], rt)                                # [(b, c), (d, e)]
                outer = outer.view(b1 - b0, co, n, co).permute(0, 2, 1, 3).reshape((b1 - b0) * n, co * co)
            # (outer W + b) / (eps + coverage), added to the pair rows, in the product's epilogue
            rows = out[b0:b1].view(-1, cf)
            ops.linear(outer, p["w_out"], bias=p["b_out"], out_dtype=out.dtype, mode=ops._L.LINEAR_ROWGATE_RES,
                       gate=inv_norm[b0:b1], residual=rows, out=rows)
        return out

    def forward(self, msa: torch.Tensor, mask: torch.Tensor) -> torch.Tensor:
        if in_check_mode():
            return _check_outer_product_mean(self, msa, mask)
        return self.run(msa, mask)


class MSAAttention(HipModule):
    """nn/d_attention.py:113-156."""

    def __init__(self, *args, c_msa: int = 64, c_pair: int = 128, num_head: int = 8) -> None:
        super().__init__()
        args = drop_mesh(args)
        vals = list(args) + [c_msa, c_pair, num_head][len(args):]
        c_msa, c_pair, num_head = vals[:3]
        if c_pair != 128:
            raise ValueError("the HIP pair-logit projection is built for c_pair = 128")
        self.c_msa, self.c_pair, self.num_head = c_msa, c_pair, num_head
        self.value_dim = c_msa // num_head
        self.act_norm = nn.LayerNorm(c_msa)
        self.pair_norm = nn.LayerNorm(c_pair)
        self.pair_logits = nn.Linear(c_pair, num_head, bias=False)
        self.v_projection = nn.Linear(c_msa, c_msa, bias=False)
        self.gating_query = nn.Linear(c_msa, c_msa, bias=False)
        self.output_projection = nn.Linear(c_msa, c_msa, bias=False)

    @property
    def native(self) -> bool:
        return self.c_msa == 64 and self.num_head == 8

    def _pack(self):
        return dict(ln_w=f32(self.act_norm.weight), ln_b=f32(self.act_norm.bias),
                    pn_w=f32(self.pair_norm.weight), pn_b=f32(self.pair_norm.bias),
                    w_logits=pad_rows(bf16(self.pair_logits.weight), 32), w_v=bf16(self.v_projection.weight),
                    w_g=bf16(self.gating_query.weight), w_o=bf16(self.output_projection.weight))

    def block(self) -> "L.MsaBlockStruct":
        """The packed weights as the library's structure."""
        d = self.packed()
        if self._native is None or self._native[1] is not d:
            s = L.MsaBlockStruct()
            point(s, ("ma_ln_w", d["ln_w"], (64,)), ("ma_ln_b", d["ln_b"], (64,)), ("ma_pn_w", d["pn_w"], (128,)),
                  ("ma_pn_b", d["pn_b"], (128,)), ("ma_w_logits", d["w_logits"], (32, 128)),
                  *((f"ma_{k}", d[k], (64, 64)) for k in ("w_v", "w_g", "w_o")))
            s.epsilon = 1.0      # (of a coverage that this operator does not use)
            self._native = (s, d)
        return self._native[0]

    def _structures(self):
        if self.native:
            self.block()

    @torch.no_grad()
    def run(self, msa, msa_mask, pair, residual: bool):
        p = self.packed()
        a, n, c = msa.shape
        if self.native and _takes(msa, msa_mask):
            return ops.msa_attention(self.block(), msa.contiguous(), msa_mask, pair.contiguous(), residual)
        h, d = self.num_head, self.value_dim
        x = ops.layer_norm(msa.contiguous(), p["ln_w"], p["ln_b"])
        logits = ops.pair_logits(pair.contiguous(), p["pn_w"], p["pn_b"], p["w_logits"], h)     # [h, q, k] fp32
        # softmax over the keys of logits + 1e9 (key mask - 1), bf16, rows padded to a multiple of 8
        w = ops.masked_softmax_rows(logits, msa_mask.float().max(dim=0).values.contiguous())        # [h, q, k]
        if n % 8 == 0 and c % 8 == 0:
            # Everything with the tokens innermost: the value and gate projections are taken
            # transposed (weights as the left operand), [(h, d), (row, k)], which is per head the
            # k-contiguous right operand of the averaging product; its result [(h, d), (row, q)]
            # has the same layout, takes the gate there and is transposed once for the output projection.
            x2 = x.view(a * n, c)
            v_t = ops.linear(p["w_v"], x2)                                                        # [(h d), (row, k)]
            gate_t = ops.linear(p["w_g"], x2, sigmoid=True)
            avg_t = ops.batched_nt_product(v_t.view(h, d * a, n), w)                              # [h, (d, row), q]
            avg = ops.transpose2d(avg_t.view(c, a * n) * gate_t).view(a, n, c)
        else:
            v = ops.linear(x, p["w_v"])                                                           # [a, k, (h d)]
            gate = ops.linear(x, p["w_g"], sigmoid=True)
            vt = _pad_last(v.view(a, n, h, d).permute(2, 0, 3, 1).reshape(h, a * d, n)).contiguous()
            avg = ops.batched_nt_product(w, vt)                                                   # [h, q, (row, d)]
            avg = avg.view(h, n, a, d).permute(2, 1, 0, 3).reshape(a, n, c) * gate
        if residual:
            return ops.linear(avg, p["w_o"], out_dtype=msa.dtype, mode=ops._L.LINEAR_GATE_RES, residual=msa, out=msa)
        return ops.linear(avg, p["w_o"], out_dtype=msa.dtype)

    def forward(self, msa: torch.Tensor, msa_mask: torch.Tensor, pair: torch.Tensor) -> torch.Tensor:
        if in_check_mode():
            return _check_msa_attention(self, msa, msa_mask, pair)
        return self.run(msa, msa_mask, pair, residual=False)


class EvoformerBlock(HipModule):
    """nn/d_pairformer.py:174-252."""

    def __init__(self, *args, c_msa: int = 64, c_pair: int = 128, n_heads_pair: int = 4) -> None:
        super().__init__()
        args = drop_mesh(args)
        vals = list(args) + [c_msa, c_pair, n_heads_pair][len(args):]
        c_msa, c_pair, n_heads_pair = vals[:3]
        self.c_msa, self.c_pair = c_msa, c_pair
        self.outer_product_mean = OuterProductMean(c_msa=c_msa, num_output_channel=c_pair)
        self.msa_attention1 = MSAAttention(c_msa=c_msa, c_pair=c_pair)
        self.msa_transition = Transition(c_x=c_msa)
        self.triangle_multiplication_outgoing = TriangleMultiplication(c_pair=c_pair, _outgoing=True)
        self.triangle_multiplication_incoming = TriangleMultiplication(c_pair=c_pair, _outgoing=False)
        self.pair_attention1 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=False)
        self.pair_attention2 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=True)
        self.pair_transition = Transition(c_x=c_pair)

    def _pack(self):
        return {}

    def _tracks(self):
        m = self._modules
        return ((m["outer_product_mean"], m["msa_attention1"], m["msa_transition"]),
                (m["triangle_multiplication_outgoing"], m["triangle_multiplication_incoming"], m["pair_attention1"],
                 m["pair_attention2"], m["pair_transition"]))

    @property
    def one_call(self) -> bool:
        """Whether the whole block runs as one call of the library (`native`)."""
        (opm, att, transition), track = self._tracks()
        return (as_written((opm, OuterProductMean), (att, MSAAttention), (transition, Transition)) and opm.native and att.native
                and transition.narrow and plain_pair_track(*track, self.c_pair) and track[2].fused)

    def _structures(self):
        if self.one_call:
            self.native()

    def native(self) -> "L.MsaBlockStruct":
        """The packed weights of the block's modules as the library's structure; made again when any of them has been
        packed again."""
        msa_track, track = self._tracks()
        packs = packs_of(msa_track + track)
        if self._native is not None and all(map(operator.is_, self._native[1], packs)):
            # (an attribute like any other, not a packed weight: as it is at the call)
            self._native[0].epsilon = self.outer_product_mean.epsilon
            return self._native[0]
        s = L.MsaBlockStruct()
        for prefix, src in (("opm_", msa_track[0].block()), ("ma_", msa_track[1].block())):
            if s.device not in (None, src.device):
                raise ValueError(f"weights of the block on {s.device} and on {src.device}")
            s.device = src.device
            for name, _ in s._fields_:
                if name.startswith(prefix):
                    setattr(s, name, getattr(src, name))
        s.epsilon = self.outer_product_mean.epsilon
        t = packs[2]
        s.mt_hidden = t["w2_64"].shape[1]
        point(s, ("mt_ln_w", t["ln_w64"], (64,)), ("mt_ln_b", t["ln_b64"], (64,)), ("mt_w1", t["w1_64"], (2 * s.mt_hidden, 64)),
              ("mt_w2", t["w2_64"], (64, s.mt_hidden)))
        p = L.PairformerBlockStruct()
        p.device = s.device
        frags = fill_pair_weights(p, *track, self.c_pair)
        s.pair = p
        self._native = (s, packs, frags)
        return s

    @torch.no_grad()
    def forward(self, msa: torch.Tensor, pair: torch.Tensor, msa_mask: torch.Tensor, pair_mask: torch.Tensor):
        """msa [rows, N, c_msa], pair [N, N, c_pair], msa_mask [rows, N],
        pair_mask [N, N] -> (msa, pair), both updated in place."""
        if in_check_mode():
            pair = pair + self.outer_product_mean(msa, msa_mask)
            msa = msa + self.msa_attention1(msa, msa_mask, pair)
            msa = msa + self.msa_transition(msa)
            pair = pair + self.triangle_multiplication_outgoing(pair, pair_mask)
            pair = pair + self.triangle_multiplication_incoming(pair, pair_mask.t().contiguous())
            pair = pair + self.pair_attention1(pair, pair_mask)
            pair = pair + self.pair_attention2(pair, pair_mask)
            pair = pair + self.pair_transition(pair)
            return msa, pair
        if not (pair.is_contiguous() and msa.is_contiguous()):
            raise ValueError("msa and pair must be contiguous (they are updated in place)")
        if self.one_call and _takes(msa, msa_mask):
            ops.evoformer_stack([self.native()], msa, pair, msa_mask, pair_mask)
            return msa, pair
        self.outer_product_mean.run(msa, msa_mask, residual=pair)
        self.msa_attention1.run(msa, msa_mask, pair, residual=True)
        self.msa_transition.run(msa, residual=True)
        self.triangle_multiplication_outgoing.run(pair, pair_mask, residual=True)
        self.triangle_multiplication_incoming.run(pair, pair_mask.t().contiguous(), residual=True)   # :217
        self.pair_attention1.run(pair, pair_mask, residual=True)
        self.pair_attention2.run(pair, pair_mask, residual=True)
        self.pair_transition.run(pair, residual=True)
        return msa, pair


def evoformer_loop(blocks, msa, pair, msa_mask, pair_mask):
    """Run Evoformer blocks one after the other (d_alphafold3.py:228-231), in one call where they allow it."""
    blocks = list(blocks)
    if (not in_check_mode() and pair.is_cuda and len(blocks) > 1 and msa.is_contiguous() and pair.is_contiguous()
            and _takes(msa, msa_mask) and all(as_written((b, EvoformerBlock)) and b.one_call and
                    b.outer_product_mean.epsilon == blocks[0].outer_product_mean.epsilon for b in blocks)):
        ops.evoformer_stack([b.native() for b in blocks], msa, pair, msa_mask, pair_mask)
        return msa, pair
    for blk in blocks:
        msa, pair = blk(msa=msa, pair=pair, msa_mask=msa_mask, pair_mask=pair_mask)
    return msa, pair


# ------------------------------------------------------------ fp32 check mode

def _check_outer_product_mean(mod: OuterProductMean, msa, mask):
    m = mask.float()[..., None]
    x = check._ln(msa.float().contiguous(), mod.layer_norm_input)
    left = m * check._lin(x, mod.left_projection)
    right = m * check._lin(x, mod.right_projection)
    a, n, co = left.shape
    lt = left.permute(1, 2, 0).reshape(n * co, a).contiguous()
    rt = right.permute(1, 2, 0).reshape(n * co, a).contiguous()
    outer = ops.ck_linear(lt, rt).view(n, co, n, co).permute(0, 2, 1, 3).reshape(n * n, co * co).contiguous()
    w = mod.output_w.detach().float().reshape(co * co, -1).t().contiguous()
    act = ops.ck_linear(outer, w, bias=mod.output_b.detach().float().contiguous()).view(n, n, -1)
    norm = (mask.float().t() @ mask.float())[..., None]
    return act / (mod.epsilon + norm)


def _check_msa_attention(mod: MSAAttention, msa, msa_mask, pair):
    a, n, c = msa.shape
    h, d = mod.num_head, mod.value_dim
    x = check._ln(msa.float().contiguous(), mod.act_norm)
    z = check._ln(pair.float().contiguous(), mod.pair_norm)
    logits = check._lin(z, mod.pair_logits).permute(2, 0, 1)
    logits = logits + 1e9 * (msa_mask.float().max(dim=0).values - 1.0)
    w = torch.softmax(logits, dim=-1).contiguous()
    v = check._lin(x, mod.v_projection)
    vt = v.view(a, n, h, d).permute(2, 0, 3, 1).reshape(h, a * d, n).contiguous()
    avg = torch.stack([ops.ck_linear(w[i], vt[i]) for i in range(h)])
    avg = avg.view(h, n, a, d).permute(2, 1, 0, 3).reshape(a, n, c)
    avg = (avg * torch.sigmoid(check._lin(x, mod.gating_query))).contiguous()
    return check._lin(avg, mod.output_projection)
