"""ctypes binding of libohara_decode.so (declared in include/ohara_decode.h).

The HIP library is the only compute path of this package: if it has not been built
(``python -m ohara_amd.build``) loading fails loudly; there is no eager/CPU fallback.
"""

from __future__ import annotations

import ctypes as C
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libohara_decode.so")
# fewer sources, the same entry points where present: what ohara_amd.build.ensure built, loaded if the full library is not built
partial_path = None

OK, EINVAL, ELAUNCH, ESIZE = 0, -1, -2, -3
_ERR = {EINVAL: "invalid argument", ELAUNCH: "HIP launch failed", ESIZE: "size not supported"}

EPI_STORE, EPI_RESIDUAL, EPI_SWIGLU = 0, 1, 2

_p, _i, _f, _i64 = C.c_void_p, C.c_int, C.c_float, C.c_int64


class OharaLayer(C.Structure):
    _fields_ = [("wqkv", _p), ("wo", _p), ("wgu", _p), ("wdown", _p), ("norm1", _p), ("norm2", _p)]


class OharaModel(C.Structure):
    _fields_ = [
        ("n_layers", _i), ("d_model", _i), ("n_heads", _i), ("n_kv_heads", _i), ("head_dim", _i),
        ("d_ff", _i), ("vocab", _i), ("t_max", _i),
        ("eps", _f), ("reserved", _i),
        ("token_emb", _p), ("final_norm", _p), ("w_vocab", _p), ("cos", _p), ("sin", _p),
        ("layers", C.POINTER(OharaLayer)),
    ]


class OharaBitLayer(C.Structure):
    _fields_ = [("w", _p * 7), ("norm_w", _p * 7), ("gamma", _f * 7), ("reserved", _f), ("norm1", _p), ("norm2", _p)]


class OharaBitModel(C.Structure):
    _fields_ = [
        ("n_layers", _i), ("d_model", _i), ("n_heads", _i), ("n_kv_heads", _i), ("head_dim", _i),
        ("d_ff", _i), ("vocab", _i), ("t_max", _i),
        ("eps", _f), ("reserved", _i),
        ("token_emb", _p), ("final_norm", _p), ("w_vocab", _p), ("cos", _p), ("sin", _p),
        ("layers", C.POINTER(OharaBitLayer)),
    ]


class OharaDecodeState(C.Structure):
    _fields_ = [
        ("batch", _i), ("rows_cap", _i), ("n_split", _i), ("valid_vocab", _i), ("hist_cap", _i), ("prof_kernel", _i),
        ("ids", _p), ("x", _p), ("q", _p), ("attn", _p), ("act", _p), ("xn", _p), ("logits", _p),
        ("attn_ws", _p), ("step_state", _p), ("history", _p),
        ("kcache", C.POINTER(_p)), ("vcache", C.POINTER(_p)),
        ("kv_int8", _i), ("kvstats", C.POINTER(_p)), ("kstage", _p), ("vstage", _p), ("kdeq", _p), ("vdeq", _p),
        ("seq_pos", _p), ("prof_start", _p), ("prof_stop", _p),
    ]


class OharaMoeLayer(C.Structure):
    _fields_ = [
        ("wqkv", _p), ("wo", _p), ("norm1", _p), ("norm2", _p), ("wgu", _p), ("wdown", _p), ("router", _p), ("router_bias", _p),
        ("experts_gu", _p), ("experts_down", _p), ("gu_stride", _i64), ("down_stride", _i64), ("counter", _p),
        ("ff", _i), ("n_experts", _i), ("hidden", _i), ("k", _i), ("biased_topk", _i), ("gate_sigmoid", _i), ("normalize", _i),
        ("reserved", _i),
    ]


class OharaMoeCall(C.Structure):
    _fields_ = [
        ("n_layers", _i), ("d_model", _i), ("n_heads", _i), ("n_kv_heads", _i), ("head_dim", _i), ("vocab", _i), ("t_max", _i),
        ("batch", _i), ("seq_len", _i), ("pos", _i), ("n_split", _i), ("last_only", _i), ("eps", _f), ("reserved", _i),
        ("token_emb", _p), ("final_norm", _p), ("w_vocab", _p), ("cos", _p), ("sin", _p), ("layers", C.POINTER(OharaMoeLayer)),
        ("ids", _p), ("kcache", C.POINTER(_p)), ("vcache", C.POINTER(_p)), ("kvstats", C.POINTER(_p)), ("logits", _p),
        ("attn_ws", _p), ("scratch", _p), ("scratch_bytes", _i64),
    ]


class OharaSeq(C.Structure):
    _fields_ = [("batch", _i), ("seq_len", _i), ("pos", _i), ("pos_stride", _i), ("pos_dev", _p), ("lens", _p), ("slots", _p)]


class OharaDelta(C.Structure):
    _fields_ = [
        ("heads", _i), ("kv_heads", _i), ("dim", _i), ("vdim", _i), ("taps", _i), ("rank_a", _i), ("rank_g", _i),
        ("off_a", _i), ("off_g", _i), ("off_b", _i), ("eps", _f), ("flags", _i),
        ("conv_w", _p), ("a2", _p), ("g2", _p), ("neg_a", _p), ("dt_bias", _p), ("norm_w", _p),
    ]


class OharaScores(C.Structure):
    _fields_ = [("scale", _f), ("cap", _f), ("chunk", _i), ("gate_elements", _i), ("ld_k", _i), ("ld_v", _i), ("slopes", _p),
                ("sinks", _p), ("window", _i), ("out_scale", _f), ("k_shared", _p), ("ld_shared", _i), ("d_shared", _i), ("ld_q", _i),
                ("reserved", _i)]


class OharaMixedScores(C.Structure):
    _fields_ = [("scale", _f), ("window", _i), ("keep", _i), ("reserved", _i), ("temp", _p), ("talk", _p)]


class OharaMixture(C.Structure):
    _fields_ = [("top", _i), ("experts", _i), ("ldy", _i), ("ldh", _i), ("lds", _i), ("reserved", _i), ("w", _p), ("idx", _p),
                ("pos_of", _p), ("y", _p), ("h", _p), ("shared", _p)]


class OharaGlu(C.Structure):
    _fields_ = [("limit", _f), ("alpha", _f), ("offset", _f), ("reserved", _i)]


class OharaRetention(C.Structure):
    _fields_ = [("heads", _i), ("dim", _i), ("vdim", _i), ("vdim_used", _i), ("off_q", _i), ("off_k", _i), ("off_v", _i), ("off_g", _i),
                ("eps", _f), ("k_scale", _f), ("out_scale", _f), ("reserved", _i), ("powers", _p)]


OUT_NONE, OUT_COPY, OUT_CONV, OUT_NORM = 0, 1, 2, 3
CENTER_Y, CENTER_OUT = 16, 32
DELTA_SILU_GATE = 1
ROUTER_SIGMOID, ROUTER_PLAIN = 1, 2
RETENTION_CHUNK = 128
OHARA_LOGITS_NONE, OHARA_LOGITS_LAST, OHARA_LOGITS_ALL = 0, 1, 2

_PROTOS = {
    "ohara_abi_version": (_i, []),
    "ohara_pack_rows_bf16": (_i, [_p, _i, _i, _i, _p, _i, _p, C.POINTER(_i64), _p]),
    "ohara_swiglu_perm": (_i, [_i, _p]),
    "ohara_embed_bf16": (_i, [_p, _p, _p, _i, _i, _i, _p]),
    "ohara_rmsnorm_bf16": (_i, [_p, _p, _p, _i, _i, _f, _p]),
    "ohara_linear_bias_add2_bytes": (_i64, [_i, _i, _i]),
    "ohara_linear_bias_add2_bf16": (_i, [_p, _i, _p, _i, _i, _p, _i, _p, _i, _p, _i, _p, _i, _p, _i64, _p]),
    "ohara_gemm_residual_norm_bytes": (_i64, [_i, _i, _i]),
    "ohara_gemm_residual_norm_bf16": (_i, [_p, _i, _p, _i, _i, _i, _p, _p, _f, _p, _p, _i64, _p]),
    "ohara_gemm_skinny_bf16": (_i, [_p, _i, _p, _i, _i, _p, _f, _i, _i, _p, _i, _p, _i, _p]),
    "ohara_projection_norm_ahead": (_i, [_i, _i, _i]),
    "ohara_gemm_tile_of": (_i, [_i, _i, _i]),
    "ohara_gemm_tile_with": (_i, [_i, _i, _i, _i, _i]),
    "ohara_gemm_first_rows": (_i, [_i, _i, _i, _i, _i]),
    "ohara_gemm_bf16": (_i, [_p, _i, _p, _i, _i, _i, _i, _p, _i, _p, _i, _p]),
    "ohara_qkv_rope_append_bf16": (_i, [_p, _i, _p, _i, _p, _f, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_qkv_rope_bf16": (_i, [_p, _i, _p, _i, _p, _f, _i, _i, _i, _i, _i, _p, _p, _i, _p, _i, _p, _p, _p, _p]),
    "ohara_kv_quant_append_int8": (_i, [_p, _p, _i, _i, _i, _i, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_kv_dequant_int8": (_i, [_p, _p, _i, _i, _i, _i, _i, _i, _p, _p]),
    "ohara_attn_append_int8": (_i, [_p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _i, _i, _p, _p, _p]),
    "ohara_attn_cached_int8": (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_attn_workspace_bytes": (_i64, [_i, _i, _i, _i, _i]),
    "ohara_attn_cached_bf16": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_attn_cached_bf16_noalloc": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p]),
    "ohara_qkv_rope_ragged_bf16": (_i, [_p, _i, _p, _i, _p, _f, _i, _i, _i, _i, _i, _p, _p, _p, _i, _p, _p, _p, _p]),
    "ohara_kv_quant_append_ragged_int8": (_i, [_p, _p, _i, _i, _i, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_attn_cached_ragged_int8": (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_attn_cached_ragged_bf16": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_qkv_rope_append_ragged_bf16": (_i, [_p, _i, _p, _i, _p, _f, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _p, _i, _p]),
    "ohara_advance_positions": (_i, [_p, _p, _i, _i, _p]),
    "ohara_advance_ragged": (_i, [_p, _p, _p, _p, _i, _i, _p]),
    "ohara_set_slots": (_i, [_p, _p, _i, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_qkv_rope_append_rows_bf16": (_i, [_p, _i, _p, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _p, _i, _p]),
    "ohara_attn_prompts_bf16": (_i, [_p, _p, _p, _i, _p, _p, _i, _i, _i, _i, _p, _p]),
    "ohara_attn_prefill_wins": (_i, [_i, _i, _i, _i, _i, _i]),
    "ohara_attn_prefill_wins_with": (_i, [_i, _i, _i, _i, _i, _i, _i64]),
    "ohara_attn_prefill_ws_bytes": (_i64, [_i, _i, _i, _i, _i, _i]),
    "ohara_attn_prefill_ws_bf16": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _p, _i64, _p]),
    "ohara_attn_prefill_bf16": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _p]),
    "ohara_argmax_bf16": (_i, [_p, _i, _i, _i, _i, _p, _p, _i, _p, _p]),
    "ohara_sample_topk_topp": (_i, [_p, _i, _i, _i, _i, _i, _f, _i, _f, _p, _i, _p, _p, _i, _p, _p]),
    "ohara_sample_topk_topp_exclusive": (_i, [_p, _i, _i, _i, _i, _i, _f, _i, _f, _p, _i, _p, _p, _i, _p, _p]),
    "ohara_sample_workspace_bytes": (_i64, []),
    "ohara_sample_topk_topp_ws": (_i, [_p, _i, _i, _i, _i, _i, _f, _i, _f, _p, _i, _p, _p, _i, _p, _p, _i64, _p]),
    "ohara_bitlinear_pack_ternary": (_i, [_p, _i, _i, _i, _p, C.POINTER(_i64), _p]),
    "ohara_act_quant_int8": (_i, [_p, _i, _p, _f, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_gemv_ternary_i8": (_i, [_p, _i, _p, _p, _p, _i, _i, _f, _i, _p, _i, _p, _i, _p, _i, _p]),
    "ohara_act_quant_swiglu_int8": (_i, [_p, _p, _i, _p, _f, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_act_quant_sets_int8": (_i, [_p, _i, _p, _p, _i, _f, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_gemm_ternary_sets_i8": (_i, [_p, _i, _p, _p, _p, _p, _i, _i, _i, _i, _p, _i, _p]),
    "ohara_gemm_ternary_qkv_rope_append": (_i, [_p, _i, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _p, _p, _i,
                                                _p]),
    "ohara_bitlinear_bf16": (_i, [_p, _i, _p, _p, _f, _p, _i, _i, _f, _i, _p, _i, _p, _i, _p, _i, _p]),
    "ohara_bitlinear_qkv_rope_append_bf16": (_i, [_p, _i, _p, _f, _i, _p, _p, _p, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _p,
                                                  _p, _i, _p]),
    "ohara_bitlinear_gate_up_bf16": (_i, [_p, _i, _p, _f, _i, _i, _p, _p, _f, _p, _p, _f, _i, _p, _i, _p]),
    "ohara_silu_mul_bf16": (_i, [_p, _p, _p, _i64, _p]),
    "ohara_rope_append_bf16": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _p, _i, _p]),
    "ohara_moe_route_topk": (_i, [_p, _i, _p, _i, _i, _i, _i, _i, _i, _p, _p, _p]),
    "ohara_moe_sort_pairs": (_i, [_p, _i, _i, _p, _p, _p, _p]),
    "ohara_moe_experts_gate_up": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _p, _p, _p, _i, _p]),
    "ohara_moe_experts_down": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_moe_route_fused": (_i, [_p, _i, _p, _f, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p, _i, _p, _p, _p, _p, _p,
                                   _p, _p]),
    "ohara_moe_experts_gate_up_shared": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _p, _p, _p, _i, _p, _i, _i, _p, _i, _p]),
    "ohara_moe_experts_down_shared": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _p, _p, _p, _p, _i, _p, _i, _i, _p, _i, _p, _i,
                                           _p]),
    "ohara_moe_experts_gate_up_many": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _i, _p, _p, _p, _i, _p]),
    "ohara_moe_experts_down_many": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _i, _p, _p, _p, _p, _i, _p]),
    "ohara_moe_forward_bytes": (_i64, [_p]),
    "ohara_moe_forward": (_i, [_p, _p]),
    "ohara_moe_combine": (_i, [_p, _i, _p, _p, _i, _i, _p, _i, _p, _i, _p, _i, _i, _p]),
    "ohara_llama_prompts": (_i, [C.POINTER(OharaModel), C.POINTER(OharaDecodeState), _i, _p, _p, _p]),
    "ohara_llama_forward": (_i, [C.POINTER(OharaModel), C.POINTER(OharaDecodeState), _i, _i, _i, _i, _i, _p]),
    "ohara_linear_bias_bf16": (_i, [_p, _i, _p, _i, _i, _p, _i, _i, _p, _i, _p, _i, _p, _i, _p]),
    "ohara_phi_block_norms": (_i, [_i, _i, _i]),
    "ohara_phi_block_in_bf16": (_i, [_p, _i, _p, _p, _f, _p, _p, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _i, _p, _i, _p]),
    "ohara_layernorm_bf16": (_i, [_p, _i, _p, _p, _p, _i, _i, _i, _f, _p]),
    "ohara_kv_append_bf16": (_i, [_p, _p, _i, _i, _i, _i, _i, _i, _p, _p, _p, _i, _p]),
    "ohara_phi_attn_workspace_bytes": (_i64, [_i, _i, _i, _i]),
    "ohara_phi_attn_bf16": (_i, [_p, _i, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p]),
    "ohara_phi_attn_linear_bf16": (_i, [_p, _i, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _p, _i, _p, _i, _i, _p, _p, _i, _p]),
    "ohara_phi_prefill_teams": (_i, [_i, _i, _i, _i]),
    "ohara_phi_attn_linear_chunks": (_i, [_i, _i, _i, _i, _i, _i, _i]),
    "ohara_phi_attn_out_bf16": (_i, [_p, _i, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _i, _p, _p, _i, _p, _i, _i, _p, _p, _i, _p, _p, _p, _i, _p, _i, _p]),
    "ohara_phi_attn_out_chunks": (_i, [_i, _i, _i, _i, _i, _i, _i, _i]),
    "ohara_persistent_workspace_bytes": (_i64, [C.POINTER(OharaModel), _i, _i, _i]),
    "ohara_persistent_barrier_offset": (_i64, [C.POINTER(OharaModel), _i, _i, _i]),
    "ohara_persistent_polled": (_i, [C.POINTER(OharaModel), _i, _i]),
    "ohara_persistent_error_offset": (_i64, [C.POINTER(OharaModel), _i, _i, _i]),
    "ohara_persistent_profile_offset": (_i64, [C.POINTER(OharaModel), _i, _i, _i]),
    "ohara_llama_decode_persistent": (_i, [C.POINTER(OharaModel), C.POINTER(OharaDecodeState), _p, _i, _i, _i,
                                           C.c_uint, _p]),
    "ohara_bitnet_persistent_workspace_bytes": (_i64, [C.POINTER(OharaBitModel), _i, _i]),
    "ohara_bitnet_persistent_error_offset": (_i64, [C.POINTER(OharaBitModel), _i, _i]),
    "ohara_bitnet_persistent_profile_offset": (_i64, [C.POINTER(OharaBitModel), _i, _i]),
    "ohara_bitnet_decode_persistent": (_i, [C.POINTER(OharaBitModel), C.POINTER(OharaDecodeState), _p, _i, _i, _i,
                                            C.c_uint, _p]),
    **{f"ohara_{name}_{dt}": proto for dt in ("bf16", "f32") for name, proto in {
        "residual_norm": (_i, [_p, _i, _p, _p, _i, _f, _p, _i, _p, _i, _f, _i, _p, _i, _p, _p, _i, _p, C.POINTER(OharaMixture),
                               C.POINTER(OharaSeq), _p]),
        "input_conv": (_i, [_p, _i, _p, _i, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "conv_ring_store": (_i, [_p, _i, _i, _i, _p, C.POINTER(OharaSeq), _p]),
        "qkv_norm_append": (_i, [_p, _i, _i, _i, _i, _i, _p, _p, _f, _p, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "attn_bias": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, _f, _p, _p, _i, _i, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "attn_scored": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, C.POINTER(OharaScores), _p, _i, _i, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "qkv_rotate_append": (_i, [_p, _i, _i, _i, _i, _i, _p, _p, _i, _p, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "qkv_headnorm_rotate_append": (_i, [_p, _i, _i, _i, _i, _i, _p, _p, _f, _p, _p, _i, _p, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "retention_step": (_i, [C.POINTER(OharaRetention), _p, _i, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "retention_prefill": (_i, [C.POINTER(OharaRetention), _p, _i, _p, _p, _i64, _p, _i, C.POINTER(OharaSeq), _p]),
        "moe_router": (_i, [_p, _i, _p, _i, _p, _i, _i, _i, _i, _i, _i, _i, _p, _p, _p, _p, _p, _p, _p, _p]),
        "gemm_gelu_lookup": (_i, [_p, _i, _p, _i, _i, _p, _i, _p, _i, _i, _p, _i, _p]),
        "latent_front": (_i, [_p, _i, _i, _i, _i, _p, _p, _f, _p, _p, _i, _p, C.POINTER(OharaSeq), _p]),
        "latent_rotary_front": (_i, [_p, _i, _i, _i, _i, _p, _p, _p, _i, _i, _i, _i, _i, _p, _f, _p, _i, _p, C.POINTER(OharaSeq), _p]),
        "head_linear": (_i, [_p, _i, _p, _i, _i, _i, _i, _i, _p, _i, _p, _i, _i, _i, _p]),
        "attn_mixed": (_i, [_p, _p, _p, _i, _i, _i, _i, _i, C.POINTER(OharaMixedScores), _i, _i, _p, _i64, _p, _i, C.POINTER(OharaSeq), _p]),
        "attn_latent": (_i, [_p, _p, _i, _i, _i, _i, _f, _i, _i, _p, _p, C.POINTER(OharaSeq), _p]),
        "delta_step": (_i, [C.POINTER(OharaDelta), _p, _i, _p, _p, _p, _i, C.POINTER(OharaSeq), _p]),
        "delta_prefill": (_i, [C.POINTER(OharaDelta), _p, _i, _p, _i, _p, _i, _p, _p, _p, _i64, _p, _p, _i,
                               C.POINTER(OharaSeq), _p]),
    }.items()},
    "ohara_gemm_glu_bf16": (_i, [_p, _i, _p, _i, _i, _f, _f, _f, _i, _p, _i, _p]),
    "ohara_gemm_xielu_bf16": (_i, [_p, _i, _p, _i, _i, _p, _f, _f, _i, _p, _i, _p]),
    "ohara_gemm_xielu_f32": (_i, [_p, _i, _p, _i, _i, _p, _f, _f, _i, _p, _i, _p]),
    "ohara_gemm_glu_f32": (_i, [_p, _i, _p, _p, _i, _i, _f, _f, _f, _i, _p, _i, _p]),
    "ohara_moe_glu_bf16": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _i, _p, _p, _p, C.POINTER(OharaGlu), _p, _i, _p, _i, _i,
                                C.POINTER(OharaGlu), _p, _i, _p]),
    "ohara_moe_down_bf16": (_i, [_p, _i, _p, _i64, _i, _i, _i, _i, _p, _p, _i, _p, _i, _i, _p, _i, _p, _i, _p]),
    "ohara_moe_glu_f32": (_i, [_p, _i, _p, _p, _i, _i, _i, _i, _i, _p, _p, _p, C.POINTER(OharaGlu), _p, _i, _p]),
    "ohara_moe_down_f32": (_i, [_p, _i, _p, _i, _i, _i, _i, _p, _p, _i, _p]),
    "ohara_retention_workspace_bytes": (_i64, [_i, _i, _i, _i, _i]),
    "ohara_gemm_f32": (_i, [_p, _i, _p, _p, _p, _f, _i, _i, _i, _p, _i, _p]),
    "ohara_gemm_softcap_bf16": (_i, [_p, _i, _p, _i, _i, _f, _i, _p, _i, _p]),
    "ohara_token_side_bf16": (_i, [_p, _i, _p, _i, _p, _i, _p, _p, _i, _p, _i, _p, _i, _p, _f, _p, _i, _i, _i, _p, _i, _p]),
    "ohara_attn_bias_workspace_bytes": (_i64, [_i, _i, _i, _i]),
    "ohara_attn_mixed_workspace_bytes": (_i64, [_i] * 11),
    "ohara_attn_latent_workspace_bytes": (_i64, [_i, _i, _i, _i]),
    "ohara_delta_workspace_bytes": (_i64, [_i, _i, _i, _i, _i]),
    "ohara_event_create": (_i, [C.POINTER(_p)]),
    "ohara_event_destroy": (_i, [_p]),
    "ohara_event_record": (_i, [_p, _p]),
    "ohara_event_elapsed_ms": (_i, [_p, _p, C.POINTER(_f)]),
}

_lib = None


def lib():
    """The loaded library; raises if it was never built."""
    global _lib
    if _lib is None:
        path = LIB_PATH if os.path.exists(LIB_PATH) or partial_path is None else partial_path
        if not os.path.exists(path):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build the HIP kernels first (python -m ohara_amd.build). "
                "ohara_amd has no fallback path."
            )
        handle = C.CDLL(path)
        for name, (res, args) in _PROTOS.items():
            if path != LIB_PATH and not hasattr(handle, name):
                continue  # an entry point of another kind of model: calling it raises
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _lib = handle
    return _lib


def check(status: int, what: str) -> None:
    if status != OK:
        raise RuntimeError(f"{what}: {_ERR.get(status, 'error')} ({status})")
