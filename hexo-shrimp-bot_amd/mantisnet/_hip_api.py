"""ctypes signatures of libmantis_hip.so (include/mantis_hip.h)."""

from __future__ import annotations

import ctypes

vp = ctypes.c_void_p
i64 = ctypes.c_int64
i32 = ctypes.c_int32
f32p = ctypes.POINTER(ctypes.c_float)



class MantisSubstage(ctypes.Structure):
    """`mantis_substage` of include/mantis_hip.h: one stage of
    mantis_attention_substages (device pointers, sizes)."""

    _fields_ = [
        ("wq", vp), ("bq", vp), ("k", vp), ("v", vp), ("ldk", i64), ("ldv", i64), ("n_src", i64),
        ("bias", vp), ("n_classes", i64), ("vcls", vp), ("seg_ptr", vp), ("src", vp), ("cls", vp),
        ("n_entries", i64), ("wo", vp), ("bo", vp),
    ]


class MantisLeafBatch(ctypes.Structure):
    """`mantis_leaf_batch`: a batch's device tables and sizes."""

    _fields_ = [
        ("stone_own", vp), ("window_feat", vp), ("moves_idx", vp), ("inc_stone", vp), ("inc_window", vp),
        ("inc_class", vp), ("stone_slot", vp), ("window_slot", vp), ("legal_offsets", vp), ("cell_pos", vp),
        ("cell_nearest", vp), ("radius_src", vp), ("radius_dst", vp), ("radius_orbit", vp), ("radius_own", vp),
        ("radius_on_axis", vp), ("dec_cell", vp), ("dec_window", vp), ("dec_class", vp), ("act_class", vp),
        ("act_rev", vp), ("act_empty", vp), ("attn_valid", vp), ("n_pos", i64), ("max_t", i64), ("max_w", i64),
        ("n_s", i64), ("n_w", i64), ("n_c", i64), ("n_cov", i64), ("n_inc", i64), ("n_rad", i64), ("n_dec", i64),
    ]


class MantisLeafBlock(ctypes.Structure):
    """`mantis_leaf_block`: one trunk block's prepared weights."""

    _fields_ = [
        ("u_w", vp), ("u_b", vp), ("mlp_w1_w", vp), ("mlp_w1_b", vp), ("mlp_w2_w", vp), ("ws_tab", vp),
        ("mlp_w3_w", vp), ("mlp_w3_b", vp), ("cr_kv_w", vp), ("cr_kv_b", vp), ("cr_q_w", vp), ("cr_q_b", vp),
        ("cr_o_w", vp), ("cr_o_b", vp), ("cr_bias", vp), ("cr_vcls", vp), ("rad_kv_w", vp), ("rad_kv_b", vp),
        ("rad_q_w", vp), ("rad_q_b", vp), ("rad_o_w", vp), ("rad_o_b", vp), ("radius_bias", vp), ("rad_vcls", vp),
        ("wr_kv_w", vp), ("wr_kv_b", vp), ("wr_q_w", vp), ("wr_q_b", vp), ("wr_o_w", vp), ("wr_o_b", vp),
        ("wr_bias", vp), ("wproj_w", vp), ("wproj_b", vp), ("mlp_s1_w", vp), ("mlp_s1_b", vp), ("mlp_s2_w", vp),
        ("mlp_s3_w", vp), ("mlp_s3_b", vp), ("qkv_w", vp), ("qkv_b", vp), ("attn_o_w", vp), ("attn_o_b", vp),
        ("lq_read_x_w", vp), ("lq_read_x_b", vp), ("lread_v_w", vp), ("lread_v_b", vp), ("lo_read_w", vp),
        ("lo_read_b", vp), ("mix_qkv_wt", vp), ("mix_qkv_b", vp), ("mix_o_wt", vp), ("mix_o_b", vp),
        ("lkv_bcast_w", vp), ("lkv_bcast_b", vp), ("bcast_q_w", vp), ("bcast_q_b", vp), ("lo_bcast_w", vp),
        ("lo_bcast_b", vp), ("ffn1_w", vp), ("ffn1_b", vp), ("ffn2_w", vp), ("ffn2_b", vp),
    ]


class MantisLeafModel(ctypes.Structure):
    """`mantis_leaf_model`: the prepared weights of mantis_leaf_forward."""

    _fields_ = [
        ("blocks", vp), ("n_blocks", i64), ("window_table", vp), ("n_patterns", i64), ("cell_table", vp),
        ("n_init", i64), ("stone_table", vp), ("latent_base", vp), ("token_moves", vp), ("sw_all", vp),
        ("n_occ", i64), ("n_dec_classes", i64), ("n_rad_classes", i64), ("ln_out_w", vp), ("ln_out_b", vp),
        ("ln_value_w", vp), ("ln_value_b", vp), ("value_queries", vp), ("mlp_v0_wt", vp), ("mlp_v0_b", vp),
        ("mlp_v2_wt", vp), ("mlp_v2_b", vp), ("n_bins", i64), ("act_proj_w", vp), ("act_proj_b", vp),
        ("head1_w", vp), ("head1_b", vp), ("head2_w", vp), ("head3_w", vp), ("head3_b", vp), ("act_table", vp),
        ("n_act", i64), ("empty_rows", vp), ("head_tab", vp), ("glin_wt", vp),
    ]


class MantisLeafOut(ctypes.Structure):
    """`mantis_leaf_out`: the outputs of mantis_leaf_forward."""

    _fields_ = [
        ("bin_centers", vp), ("rows", vp), ("policy", vp), ("q_values", vp), ("q_score", vp), ("value", vp),
        ("dist", vp), ("logits", vp),
    ]


SIGNATURES = {
    "mantis_hip_version": ([], i32),
    "mantis_plan_check": ([vp, vp, i64, vp, vp, i64, vp, i64, i64, vp, vp], i32),
    "mantis_stable_key_order_workspace": ([i64, i64], i64),
    "mantis_stable_key_count": ([vp, i64, i64, vp, vp, vp], i32),
    "mantis_stable_key_order": ([vp, vp, vp, i64, i64, vp, vp, vp, vp, vp], i32),
    "mantis_stable_key_order_noalloc": ([vp, vp, vp, i64, i64, vp, vp, vp, vp, vp], i32),
    "mantis_latent_read_x_workspace": ([i64], i64),
    "mantis_latent_read_x": ([vp, i64, vp, i64, vp, vp, i64, i64, vp, vp, vp, vp, vp, vp], i32),
    "mantis_latent_broadcast_residual": ([vp, i64, vp, i64, vp, i64, i64, vp, vp, vp, i64, vp, vp], i32),
    "mantis_latent_broadcast_project_residual": ([vp, vp, vp, i64, vp, i64, i64, vp, vp, vp, i64, vp, vp], i32),
    "mantis_covered_rows": ([vp, vp, i64, i64, vp, vp, i64, vp, vp, vp], i32),
    "mantis_window_view": ([vp, vp, vp, vp, i64, i64, i64, vp, vp, i64, vp, vp, vp, vp, vp, vp], i32),
    "mantis_radius_class": ([vp, vp, vp, i64, vp, vp], i32),
    "mantis_attention_slots": ([vp, i64, i64, i64, vp, vp, vp, vp], i32),
    "mantis_gather_rows": ([vp, i32, i64, i64, vp, vp, i64, i64, vp, i64, vp, vp], i32),
    "mantis_runs_to_ptr": ([vp, i64, i64, vp, vp, vp], i32),
    "mantis_structure_init": ([vp, vp, i64, vp, i64, vp, i64, vp, vp, i64, vp, i64, vp, i64, vp, i64, vp, vp], i32),
    "mantis_segment_order": ([vp, i64, vp, vp, i64, vp, vp, vp], i32),
    "mantis_run_reduce": ([vp, i32, i64, i64, i64, vp, i64, vp, i64, vp, i32, vp, vp], i32),
    "mantis_class_reduce_workspace": ([i64, i64, i64], i64),
    "mantis_class_reduce": ([vp, i32, i64, i64, i64, vp, i64, vp, i64, vp, i64, vp, i32, vp, vp], i32),
    "mantis_cell_pass": ([vp, i32, i64, i64, i64, vp, i32, i64, i64, vp, i64, vp, vp, i64, vp, vp, vp, vp, vp, vp],
                         i32),
    "mantis_attention_backward_workspace": ([i64, i64, i64], i64),
    "mantis_attention_backward": ([vp, vp, vp, i32, i64, i64, i64, i64, i64, vp, i64, vp, i32, vp, i64, vp, vp, vp,
                                   vp, vp, vp, i64, vp, vp, vp, vp, vp, vp, i64, vp, vp, vp, vp, vp, vp, vp], i32),
    "mantis_latent_out": ([vp, i64, vp, vp, vp, vp, vp, vp], i32),
    "mantis_value_tail": ([vp, i64, vp, vp, vp, vp, i64, vp, vp, vp, vp, vp], i32),
    "mantis_leaf_workspace": ([vp, i64], i64),
    "mantis_leaf_forward": ([vp, vp, vp, ctypes.c_float, vp, i64, vp, vp, vp, vp], i32),
    "mantis_class_order_workspace": ([i64, i64], i64),
    "mantis_class_order": ([vp, vp, i64, i64, vp, vp, vp, i64, vp, vp], i32),
    "mantis_latent_backward_workspace": ([i64, i64], i64),
    "mantis_latent_read_backward": ([vp, vp, vp, i32, i64, i64, i64, vp, vp, vp, i64, i64, vp, vp, vp, vp, vp, i64, vp,
                                     vp, vp, vp, vp], i32),
    "mantis_latent_broadcast_backward": ([vp, vp, vp, i32, i64, i64, i64, vp, vp, vp, i64, i64, vp, vp, vp, vp, i64,
                                          vp, vp, vp, vp, vp], i32),
    "mantis_row_encode_backward_workspace": ([i64, i64], i64),
    "mantis_row_encode_backward": ([vp, i32, i64, i64, vp, i32, i64, vp, i64, vp, vp, vp, i64, vp, vp, vp, vp, vp, i64,
                                    vp, vp, vp, vp], i32),
    "mantis_cell_pass_backward_workspace": ([i64, i64, i64, i64], i64),
    "mantis_cell_pass_backward": ([vp, i32, i64, i64, i64, vp, i32, i64, i64, vp, i32, i64, vp, i64, vp, vp, i64, vp,
                                   vp, vp, vp, vp, i64, vp, vp, vp, vp], i32),
    "mantis_cell_attention": (
        [vp, vp, vp, i32, i64, i64, i64, vp, i64, vp, i32, vp, vp, vp, i64, i64, i64, i32, i32, vp, i32, vp, vp, vp, vp],
        i32),
    "mantis_attention_substage": (
        [vp, i64, i64, vp, vp, vp, vp, i64, i64, i64, vp, i64, vp, vp, vp, vp, i64, vp, vp, vp, vp], i32),
    "mantis_attention_substages": ([vp, i32, i64, i64, vp, vp, i32, vp, vp, vp], i32),
    "mantis_attention_substages_init": ([vp, i32, i64, i64, vp, vp, i32, vp, i64, i64, vp, i64, vp, vp, vp], i32),
    "mantis_attention_substages_covered": ([vp, i32, i64, i64, vp, vp, vp, i64, i64, vp, i64, vp, vp, vp], i32),
    "mantis_attention_substage_project": ([vp, i32, i64, i64, vp, vp, vp, vp, vp, i64, vp, vp, vp], i32),
    "mantis_radius_chunks_capacity": ([i64, i64], i64),
    "mantis_radius_chunks": ([vp, vp, i32, i64, i64, i64, vp, i64, vp, vp, vp], i32),
    "mantis_radius_prep": ([vp, vp, i64, vp, i64, vp, vp, i64, i64, i64, vp, i64, vp, i64, vp, vp, vp, vp, vp], i32),
    "mantis_radius_stage": ([vp, i64, i64, vp, vp, vp, i64, vp, vp, vp, vp, i64, i64, vp, i64, vp, vp, i64, vp, vp,
                             vp, vp, i64, i64, vp, vp, vp], i32),
    "mantis_cell_heads": (
        [vp, i32, i32, i32, i64, i64, vp, vp, vp, vp, vp, vp, vp, i64, vp, i64, vp, vp, vp, vp, i64, vp, i64, vp, vp, vp,
         vp, vp, i64, vp, vp, vp, vp], i32),
    "mantis_improve_policy": ([vp, vp, vp, i32, vp, i64, i64, ctypes.c_double, ctypes.c_double, vp, vp, vp, vp, vp, vp],
                              i32),
    "mantis_latent_mix": ([vp, i64, i64, vp, vp, vp, vp, vp], i32),
    "mantis_latent_read": ([vp, vp, vp, i32, i64, i64, i64, vp, vp, i64, i64, i32, i32, vp, vp, vp, vp, vp, vp], i32),
    "mantis_latent_read_workspace": ([i64], i64),
    "mantis_latent_broadcast": ([vp, vp, vp, i32, i64, i64, i64, vp, i64, i64, i32, i32, vp, i32, vp, vp, vp, vp],
                                i32),
    "mantis_row_encode": ([vp, i32, i64, i64, vp, i64, vp, vp, i64, vp, i64, vp, vp, vp, vp, vp], i32),
    "mantis_stone_attention": ([vp, vp, vp, vp, vp, vp, i32, vp, i64, i32, i64, i32, vp, vp, vp, vp, vp], i32),
    "mantis_stone_attention_backward": ([vp, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp, i32, vp, i64, i32, i64, i32, vp,
                                         vp, vp, vp, vp, vp, vp, vp], i32),
    "mantis_latent_attend": ([vp, i32, i64, vp, i64, i64, vp, vp], i32),
    "mantis_stone_attention_schedule_len": ([i64, i32, i64], i64),
    "mantis_stone_attention_schedule": ([vp, i64, i32, i64, vp, vp], i32),
    "mantis_fused_linear": ([vp, i32, i64, vp, i64, i64, i32, vp, i32, i64, vp, vp, vp, i32, vp, i64, vp, vp, i64,
                             i32, vp, vp, i32, i32, vp, i64, vp, vp], i32),
    "mantis_fused_linear_split": ([vp, i32, i64, vp, i64, i64, i32, vp, i32, i64, vp, vp, vp, i32, vp, i64, vp, vp,
                                   i64, i32, vp, vp, i32, i32, vp, i64, vp, vp], i32),
    "mantis_layer_norm": ([vp, i32, i64, i64, vp, vp, vp, i32, i64, vp], i32),
    "mantis_value_read": ([vp, vp, i32, i64, vp, vp, i64, vp, vp, vp, vp, vp, i32, vp, vp, vp, vp], i32),
    "mantis_value_read_workspace": ([i64], i64),
    "mantis_compose_q": ([vp, i64, vp, i64, i64, ctypes.c_float, vp, vp, vp], i32),
    "mantis_compose_q_rows": ([vp, i64, vp, i64, i64, ctypes.c_float, vp, vp, vp, vp], i32),
    "mantis_hex_neighbours": ([vp, vp, i64, i64, vp, vp, vp], i32),
    "mantis_hex_aggregate_linear": ([vp, vp, i64, vp, vp, vp, vp, vp, vp], i32),
}


def bind(lib: ctypes.CDLL) -> ctypes.CDLL:
    for name, (args, res) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.argtypes = args
        fn.restype = res
    return lib
