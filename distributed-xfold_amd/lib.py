"""ctypes binding of libaf3hip.so (C ABI declared in include/af3_hip.h)."""

from __future__ import annotations

import ctypes as C
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libaf3hip.so")

ABI_VERSION = 4                      # AF3_ABI_VERSION: of the structures and argument lists below
AF3_BF16, AF3_F32 = 0, 1
STATIC_SCRATCH_BYTES = 32 << 20      # AF3_STATIC_SCRATCH_BYTES
LINEAR_PLAIN, LINEAR_SWIGLU, LINEAR_GATE_RES, LINEAR_REGROUP32, LINEAR_ROWGATE_RES = 0, 2, 3, 4, 5
PAIR64_MAX_TOKENS = 3072    # AF3_PAIR64_MAX_TOKENS

_vp, _i, _i64, _sz, _f = C.c_void_p, C.c_int, C.c_int64, C.c_size_t, C.c_float


class PairformerBlockStruct(C.Structure):
    """af3_pairformer_block."""
    device = None       # where what the fields point at lives (host side only, as in the other structures)
    _fields_ = (
        [(k, _vp * 2) for k in ("tm_ln_in_w", "tm_ln_in_b", "tm_ln_c_w", "tm_ln_c_b", "tm_w_proj_gate", "tm_w_out",
                                "tm_w_gating", "ta_ln_w", "ta_ln_b", "ta_w_bias", "ta_w_qkvg", "ta_w_out")]
        + [(k, _vp) for k in ("pt_ln_w", "pt_ln_b", "pt_w1", "pt_w2", "sl_ln_w", "sl_ln_b", "sl_w", "sa_ln_w", "sa_ln_b",
                              "sa_w_qkvg", "sa_q_b", "sa_w_out", "st_ln_w", "st_ln_b", "st_w1", "st_w2", "pair_frags")]
        + [(k, C.c_int32) for k in ("valid_channels", "num_head_pair", "pair_hidden", "with_single", "num_head",
                                    "c_single", "single_hidden", "pair_channels")])


class MsaBlockStruct(C.Structure):
    """af3_msa_block."""
    device = None
    _fields_ = (
        [(k, _vp) for k in ("opm_ln_w", "opm_ln_b", "opm_w_lr", "opm_w_out", "opm_b_out", "ma_ln_w", "ma_ln_b", "ma_pn_w",
                            "ma_pn_b", "ma_w_logits", "ma_w_v", "ma_w_g", "ma_w_o", "mt_ln_w", "mt_ln_b", "mt_w1", "mt_w2")]
        + [("pair", PairformerBlockStruct), ("mt_hidden", C.c_int32), ("epsilon", C.c_float)])


class DiffusionBlockStruct(C.Structure):
    """af3_diffusion_block."""
    device = None
    _fields_ = [(k, _vp) for k in ("w_q", "w_kv", "q_b", "w_out", "w_tr1", "w_tr2", "frags")]


# name -> (restype, argtypes); must list every symbol include/af3_hip.h declares
SIGNATURES = {
    "af3_abi_version": (_i, []),
    "af3_error_string": (C.c_char_p, [_i]),
    "af3_triangle_multiplication_workspace_bytes": (_sz, [_i64]),
    "af3_triangle_multiplication_forward": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _vp, _sz, _vp]),
    "af3_grid_self_attn_workspace_bytes": (_sz, [_i64, _i]),
    "af3_grid_self_attn_forward": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _vp, _sz, _vp]),
    "af3_transition_forward": (_i, [_vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _vp]),
    "af3_pair_cond_transition_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _vp]),
    "af3_row_transition_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i64, _vp]),
    "af3_triangle_multiplication_forward_padded": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i, _vp, _sz, _vp]),
    "af3_grid_self_attn_forward_padded": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _i, _vp, _sz, _vp]),
    "af3_transition_forward_padded": (_i, [_vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _i, _vp]),
    "af3_contact_matrix_forward": (_i, [_vp, _vp, _i, _vp, _vp, _i, _vp, _i64, _vp]),
    "af3_pair_embed_forward": (
        _i, [_vp, _i64, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _vp]),
    "af3_atom_embed_forward": (_i, [_vp] * 11 + [_i64, _i, _vp]),
    "af3_gather_atoms_forward": (
        _i, [_vp, _vp, _i64, _vp, _vp, _vp, _i64, _vp, _i64, _vp, _vp, _vp, _i64, _vp, _vp, _vp, _vp, _i, _vp]),
    "af3_add_rows_forward": (_i, [_vp, _vp, _i64, _i64, _vp, _i, _i64, _i, _vp]),
    "af3_mask_rows_forward": (_i, [_vp, _vp, _i64, _i64, _i, _vp]),
    "af3_augment_positions_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _vp]),
    "af3_positions_forward": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _f, _vp, _i64, _i64, _vp]),
    "af3_msa_workspace_bytes": (_sz, [_i64, _i64]),
    "af3_outer_product_mean_forward": (_i, [_vp, _vp, _i, _vp, _vp, _i, _i, _i64, _i64, _vp, _sz, _vp]),
    "af3_msa_attention_forward": (_i, [_vp, _vp, _i, _vp, _vp, _i, _vp, _i, _i64, _i64, _vp, _sz, _vp]),
    "af3_transition64_forward": (_i, [_vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _i, _i64, _vp]),
    "af3_evoformer_stack_forward": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _i, _vp, _i64, _i64, _vp, _sz, _vp, _sz, _vp]),
    "af3_batch_diffusion_self_attention_workspace_bytes": (_sz, [_i64, _i64, _i]),
    "af3_batch_diffusion_self_attention_forward": (
        _i, [_vp, _vp, _i64, _vp, _i, _vp, _vp, _i, _vp, _i, _i64, _i64, _i, _vp, _sz, _vp]),
    "af3_batch_diffusion_self_attention_forward_static": (
        _i, [_vp, _vp, _i64, _vp, _i, _vp, _vp, _i, _vp, _i, _i64, _i64, _i, _vp]),
    "af3_batched_nt_product_forward": (_i, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp]),
    "af3_transpose_bf16_forward": (_i, [_vp, _vp, _i64, _i64, _vp]),
    "af3_atom_position_features_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i64, _i64, _i64, _i, _vp]),
    "af3_gather_rows_add_forward": (_i, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _vp]),
    "af3_position_update_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _vp]),
    "af3_gathered_relu_mean_forward": (_i, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _i, _vp]),
    "af3_atom_aggregate_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _vp]),
    "af3_batch_diffusion_cross_attention_workspace_bytes": (_sz, [_i64, _i64, _i64, _i]),
    "af3_batch_diffusion_cross_attention_forward": (
        _i, [_vp, _vp, _vp, _vp, _vp, _i64, _vp, _vp, _vp, _i, _vp, _i, _i64, _i64, _i64, _i, _vp, _sz, _vp]),
    "af3_gathered_cross_attention_workspace_bytes": (_sz, [_i64, _i64, _i64, _i64, _i]),
    "af3_gathered_cross_attention_forward": (
        _i, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _vp, _vp, _vp, _i, _vp, _i, _i64, _i64, _i64, _i64, _i64, _i,
             _vp, _sz, _vp]),
    "af3_pair_logits_forward": (_i, [_vp, _i, _vp, _vp, _vp, _i, _vp, _i64, _vp]),
    "af3_pair_logits_quads_forward": (_i, [_vp, _i, _vp, _vp, _vp, _i, _vp, _i64, _vp]),
    "af3_layer_norm_forward": (_i, [_vp, _i, _vp, _i64, _i, _vp, _vp, _vp, _vp, _i64, _i64, _vp]),
    "af3_linear_forward": (
        _i, [_vp, _vp, _vp, _vp, _i, _i64, _i, _i, _i, _f, _i, _vp, _i64, _i64, _vp, _i, _vp]),
    "af3_triangle_contraction_forward": (_i, [_vp, _vp, _vp, _i64, _vp]),
    "af3_masked_softmax_rows_forward": (_i, [_vp, _vp, _vp, _i64, _i64, _i64, _vp]),
    "af3_narrow_linear_f32_forward": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _vp]),
    "af3_atom_pair_cond_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _i64, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
                                        _i64, _i64, _i64, _vp]),
    "af3_atom_pair_logits_forward": (_i, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _i, _vp]),
    "af3_atom_pair_logits_quads_forward": (_i, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i, _i, _vp]),
    "af3_pair_cond_init_forward": (_i, [_vp, _i, _f, _vp, _vp, _vp, _vp, _vp, _i, _i, _vp, _vp, _vp, _vp, _vp, _i64, _vp]),
    "af3_pairformer_stack_workspace_bytes": (_sz, [_i64, _i]),
    "af3_pairformer_single_workspace_bytes": (_sz, [_i64, _i, _i]),
    "af3_pairformer_stack_forward": (
        _i, [_vp, _i, _vp, _i, _vp, _vp, _vp, _i, _vp, _i64, _vp, _vp, _sz, _vp, _sz, _vp, _vp, _i]),
    "af3_diffusion_transformer_workspace_bytes": (_sz, [_i64, _i64, _i, _i]),
    "af3_diffusion_transformer_forward": (
        _i, [_vp, _i, _vp, _i, _i64, _i64, _i, _i, _i, _vp, _vp, _i, _vp, _vp, _i64, _vp, _sz, _vp]),
    "af3_atom_transformer_workspace_bytes": (_sz, [_i64, _i64, _i64, _i, _i]),
    "af3_atom_transformer_forward": (
        _i, [_vp, _i, _vp, _i, _i64, _i64, _i64, _i64, _i, _i, _i, _vp, _vp, _vp, _vp, _i, _vp, _vp, _vp, _vp, _sz, _vp]),
    "af3_atom_transformer_windows_forward": (
        _i, [_vp, _i, _vp, _i, _i64, _i64, _i64, _i64, _i, _i, _i, _vp, _vp, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _sz, _vp]),
    "af3_atom_windows_forward": (_i, [_vp, _vp, _vp, _i64, _vp, _i64, _i64, _i64, _vp, _vp]),
    "af3_linear_bias_span": (_i, [_i64, _i, _i, _i, _i, _vp, _vp]),
    "af3_grid_attention_core_forward": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _vp]),
    "af3_check_gemm_f32": (
        _i, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
             _vp, _f, _i, _vp, _i64, _i64, _vp, _i64, _i64, _vp]),
    "af3_check_layer_norm_f32": (_i, [_vp, _vp, _i64, _i, _vp, _vp, _vp, _vp, _i64, _i64, _vp]),
    "af3_check_elementwise_f32": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i, _vp]),
    "af3_check_attention_f32": (
        _i, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i, _i64, _i64, _i,
             _vp, _i64, _i64, _i64, _i64, _i64, _vp, _i64, _vp, _vp, _vp]),
}

_lib = None


class Af3Error(RuntimeError):
    pass


def load():
    """Load libaf3hip.so; raises if it has not been built (no fallback)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise Af3Error(
            f"{LIB_PATH} is missing: build it with `make -C {os.path.join(_HERE, 'csrc')}` "
            "(or __graft_entry__.build()); there is no CPU fallback")
    lib = C.CDLL(LIB_PATH)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)          # AttributeError if a declared symbol is absent
        fn.restype = res
        fn.argtypes = args
    if lib.af3_abi_version() != ABI_VERSION:
        raise Af3Error(f"{LIB_PATH} has interface version {lib.af3_abi_version()}, not {ABI_VERSION}: build it again")
    _lib = lib
    return lib


def check(rc: int, what: str):
    if rc != 0:
        msg = load().af3_error_string(rc).decode()
        raise Af3Error(f"{what} failed: {msg} (code {rc})")
