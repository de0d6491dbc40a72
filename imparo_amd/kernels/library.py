"""Loads the gfx950 kernel library and declares its C entry points.

The library is loaded once per process. If it has not been built yet it is
built at the first call (hipcc must be present); there is no fallback: without
the library every op raises.
"""
from __future__ import annotations

import ctypes
import os
import threading
from ctypes import c_int, c_int64, c_float, c_void_p

from ..csrc import build as _build

_lock = threading.Lock()
_lib = None

P = c_void_p
I = c_int
F = c_float

_SIGNATURES = {
    "imparo_embed_gather": [P, I, P, P, I, I, I, P],
    "imparo_place_tokens": [P, P, P, P, I, I, P],
    "imparo_rms_norm": [P, P, I, I, P, P, P, I, I, I, F, I, P],
    "imparo_gemm": [P, P, P, P, I, I, I, I, I, I, I, P],
    # x, w, bias, y, dtype, out_dtype, m, n, k, scale, limit, alpha, stream
    "imparo_gemm_gated": [P, P, P, P, I, I, I, I, I, F, F, F, P],
    "imparo_gemm_slices": [I, I, I, I],
    "imparo_gemm_adds": [I, I, I, I],
    "imparo_gemm_variant": [P, P, P, P, I, I, I, I, I, I, I, I, P],
    "imparo_short_conv_decode": [P, P, P, P, P, P, I, I, I, I, I, P],
    "imparo_in_proj_conv_decode": [P, P, P, P, P, P, P, P, I, I, I, I, I, I, P],
    "imparo_qk_norm_rope_store": [P, P, P, F, P, I, I, P, P, P, I, I, P, P, P, I, I, I, I, I, I, I, I, P],
    "imparo_attention": [P, P, P, P, I, P, P, P, I, I, I, I, I, I, I, F, I, I, P],
    "imparo_attention_decode": [P, P, P, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P],
    # qkv, q_w, k_w, eps, inv_freq, n_freq, interleaved, k_cache, v_cache, write_kv, out, part_o, part_ml, rows, n_rows,
    # seg_start, positions, table, stride, page, heads, kv_heads, head_dim, n_pages, scale, window, n_splits, stream
    "imparo_attention_decode_qkv": [P, P, P, F, P, I, I, P, P, I, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P],
    # qkv, row_ld, brings, q_w, k_w, eps, inv_freq, n_freq, interleaved, magnitude, whole, far_first, k_cache, v_cache, out, part_o,
    # part_ml, rows, n_rows, seg_start, positions, table, stride, page, heads, kv_heads, head_dim, n_pages, scale, window, n_splits, rule, stream
    "imparo_attention_decode_qkv_ruled": [P, I, I, P, P, F, P, I, I, F, I, I, P, P, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P, P],
    "imparo_attention_decode_exact": [P, P, P, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P],
    "imparo_attention_prefill_exact": [P, P, P, P, P, P, I, P, I, I, P, P, P, P, I, I, I, I, I, I, F, I, P],
    # as the exact forms, with the address of an AttentionRule before the stream
    "imparo_attention_decode_ruled": [P, P, P, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P, P],
    "imparo_attention_prefill_ruled": [P, P, P, P, P, P, I, P, I, I, P, P, P, P, I, I, I, I, I, I, F, I, P, P],
    "imparo_attention_ruled": [P, P, P, P, I, P, P, P, I, I, I, I, I, I, I, I, I, F, I, I, P, P],
    "imparo_attention_ruled_keys": [I, I, I],
    "imparo_attention_f32_split_pays": [I, I, I, I, I, I],
    "imparo_attention_decode_qkv_takes": [I, I],
    "imparo_attention_decode_qkv_pays": [I, I],
    "imparo_attention_decode_qkv_ruled_takes": [I, I, I, I, I],
    "imparo_attention_decode_qkv_ruled_pays": [I, I, I, I, I, I, I],
    "imparo_attention_prefill": [P, P, P, P, P, P, I, P, I, I, P, P, P, P, I, I, I, I, I, I, F, I, P],
    "imparo_attention_prefill_splits": [I, I, I, I, I],
    "imparo_attention_decode_split": [],
    "imparo_attention_prefill_tile": [],
    "imparo_short_conv": [P, P, P, P, P, P, P, P, I, I, I, I, I, I, P],
    "imparo_short_conv_state": [P, P, P, P, P, I, I, I, I, I, P],
    "imparo_argmax_rows": [P, P, I, I, P],
    "imparo_sample_rows": [P, P, P, P, I, I, P],
    "imparo_fill_f32": [P, F, c_int64, P],
    "imparo_fill_sites": [P, P, P, I, I, P],
    "imparo_attention_decode_static": [P, P, P, P, P, I, P, P, P, I, I, I, I, I, I, F, I, I, P],
    "imparo_load_code": [],
    "imparo_embed_sinusoid": [P, I, P, P, P, P, I, I, I, P],
    "imparo_group_rms_norm": [P, P, I, I, P, P, P, I, I, I, I, F, I, P, P, P, P],
    "imparo_token_shift": [P, P, P, P, P, P, P, P, I, I, I, I, P],
    "imparo_poly_norm": [P, I, P, P, I, I, I, I, F, P],
    "imparo_causal_conv": [P, I, P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, P],
    "imparo_selective_scan": [P, P, P, P, I, P, P, P, P, P, P, P, I, P, I, I, I, I, I, P],
    "imparo_selective_scan_chunk": [],
    "imparo_diff_qkv_store": [P, I, P, P, P, I, I, P, P, P, I, I, I, I, I, I, I, I, F, I, P],
    "imparo_diff_attention_split": [],
    # q, k_cache, v_cache, gate, gate_ld, out, part, dtype, positions, row_of_token, table, stride, page, tokens, heads,
    # kv_heads, dim, vdim, n_pages, scale, window, lambda, eps, out_scale, n_splits, stream
    "imparo_diff_attention": [P, P, P, P, I, P, P, I, P, P, P, I, I, I, I, I, I, I, I, F, I, F, F, F, I, P, I, P],
    "imparo_diff_attention_tile": [],
    "imparo_diff_attention_tiles_takes": [I, I, I],
    "imparo_diff_attention_tiles": [P, P, P, P, I, P, P, P, P, P, I, I, I, I, I, I, I, I, I, F, I, F, F, F, I, P],
    "imparo_embed_gather_scaled": [P, I, P, P, I, I, I, F, P],
    "imparo_qk_norm_rope_store_dv": [P, P, P, F, P, I, I, P, P, P, I, I, P, P, P, I, I, I, I, I, I, I, I, I, P],
    "imparo_attention_dv": [P, P, P, P, I, P, P, P, I, I, I, I, I, I, I, I, I, F, I, I, P],
    "imparo_moe_route": [P, P, P, P, I, I, I, I, I, I, I, I, F, I, P],
    # gu, weight, entry_of_slot, choice, limits, n_experts, alpha, hidden, out_dtype, n_slots, half, stream
    "imparo_moe_gated": [P, P, P, P, P, I, F, P, I, I, I, P],
    # x, in_streams, x_out, delta, n_delta, y, h, h_dtype, choice, choice_weight, slot_of_entry, top, n_experts, n_rows_x,
    # rows, streams, mix, join, read, norm, weight, bias, eps, out, out_dtype, n_out, width, stream
    "imparo_stream_norm": [P, I, P, P, I, P, P, I, P, P, P, I, I, I, P, I, P, P, P, I, P, P, F, P, I, I, I, P],
    "imparo_stream_max": [],
    "imparo_stream_step_takes": [I, I, I, I, I],
    "imparo_stream_step_pays": [I, I, I],
    "imparo_stream_step_routes": [I, I, I],
    # x, in_streams, x_out, delta, n_delta, y, h, h_dtype, choice, choice_weight, top, n_experts, n_rows, streams, mix, join, read,
    # norm, weight, bias, eps, out, out_dtype, width, router_w, router_bias, correction, n_router, route_top, scoring, normalize,
    # route_scale, always, route_choice, route_weight, stream
    "imparo_stream_step": [P, I, P, P, I, P, P, I, P, P, I, I, I, I, P, P, P, I, P, P, F, P, I, I, P, P, P, I, I, I, I, F, I, P, P, P],
    "imparo_moe_direct_takes": [I, I, I],
    "imparo_moe_direct_pays": [I, I, I, I, I],
    # a, a_ld, own_rows, choice, n_tokens, used, n_experts, w, out, out_dtype, n, k, epilogue, limits, alpha, stream
    "imparo_moe_gemm_direct": [P, I, I, P, I, I, I, P, P, I, I, I, I, P, F, P],
    # table, bigram, dtype, ids, positions, row_of_token, seg_start, seg_len, slot, state, x, n_tokens, n_rows, width, vocab,
    # n_slots, buckets, mul_prev, mul_cur, scale, advance, stream
    "imparo_embed_bigram": [P, P, I, P, P, P, P, P, P, P, P, I, I, I, I, I, I, c_int64, c_int64, F, I, P],
    # qkv, row_ld, q_w, k_w, norm, eps, inv_freq, n_freq, interleaved, magnitude, positions, row_of_token, table, stride,
    # page, q_out, k_cache, v_cache, dtype, write_kv, n_tokens, heads, kv_heads, head_dim, value_dim, n_pages,
    # v_transposed, stream
    "imparo_qk_row_norm_rope_store": [P, I, P, P, I, F, P, I, I, F, P, P, P, I, I, P, P, P, I, I, I, I, I, I, I, I, I, P],
    "imparo_attention_latent": [P, P, P, I, P, P, P, I, I, I, I, I, I, I, F, I, P],
    "imparo_latent_store": [P, P, P, F, P, I, I, P, P, P, I, I, I, P, P, P, P, I, I, I, I, I, I, P],
    "imparo_attention_latent_tiles_takes": [I, I, I],
    "imparo_attention_latent_tiles_split": [I, I, I, P],
    "imparo_attention_latent_tiles": [P, P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, F, I, I, I, I, P],
    "imparo_head_gemm": [P, I, I, P, I, P, I, I, I, I, I, I, I, P],
    "imparo_head_gemm_tiles": [P, I, I, P, P, I, I, I, I, I, I, I, P],
    "imparo_hgrn2_scan": [P, I, I, I, I, P, P, P, P, P, P, I, I, I, I, I, I, P, P, P],
    # q, ld, off, div, k, ld, off, div, v, ld, off, decay_const, step, ld, off, step_bias, rate, v_times_step, beta, ld,
    # off, skip, state, seg_start, seg_len, slot, out, n_rows, heads, dim, vdim, chunk_tokens, max_chunks, chunk_state,
    # chunk_decay, silu_in, stream
    "imparo_decay_scan": [P, I, I, I, P, I, I, I, P, I, I, P, P, I, I, P, P, I, P, I, I, P, P, P, P, P, P, I, I, I, I, I, I,
                          P, P, I, P],
    # q, ld, off, div, k, ld, off, div, v, ld, off, step, ld, off, step_bias, rate, beta, ld, off, state, seg_start,
    # seg_len, slot, out, n_rows, heads, dim, vdim, chunk_tokens, max_chunks, scratch, stream
    "imparo_channel_delta_scan": [P, I, I, I, P, I, I, I, P, I, I, P, I, I, P, P, P, I, I, P, P, P, P, P, I, I, I, I, I, I,
                                  P, P],
    "imparo_channel_delta_scratch": ([I], c_int64),
    "imparo_silu_columns": [P, I, I, I, I, P],
    # x, delta_a, n_a, delta_b, n_b, n_x_rows, rows, alpha, weight, bias, out, out_dtype, n_rows, width, write_back, stream
    "imparo_dynamic_tanh": [P, P, I, P, I, I, P, F, P, P, P, I, I, I, I, P],
    "imparo_delta_chunk_tokens": [],
    "imparo_delta_chunk_max_dim": [],
    "imparo_head_prepare": [P, I, I, I, I, I, I, F, P, I, I, P, I, F, F, P],
    "imparo_channel_delta_heads_takes": [I, I, I, I, I, I, I],
    "imparo_channel_delta_heads": [P, I, I, I, P, I, I, I, P, P, P, I, P, P, P, I, I, I, I, F, F, F, P],
    "imparo_channel_delta_step_takes": [I, I, I, I, I],
    "imparo_channel_delta_step": [P, I, I, P, I, I, P, P, I, P, P, P, I, P, P, P, I, I, I, I, I, I, F, F, F, P],
    "imparo_gated_group_norm": [P, P, I, I, P, P, I, I, I, I, F, I, I, P],
    "imparo_normed_sum": [P, I, P, P, I, P, P, I, I, F, F, P],
    "imparo_gated_row_add": [P, P, I, P, I, I, I, I, P],
    "imparo_gated_sum": [P, P, I, P, I, P, I, P, I, I, I, P],
    "imparo_side_gate": [P, P, I, I, I, P, I, P, I, I, I, I, P],
    "imparo_add_rows": [P, P, c_int64, P],
    "imparo_cast_rows": [P, P, P, I, I, I, P],
    "imparo_moe_route_plan_tokens": [],
    "imparo_moe_route_plan": [P, P, P, P, I, I, I, I, I, I, P, P, P, I, I, I, I, I, F, I, P],
    "imparo_moe_router_takes": [I, I, I, I, I, I, I],
    "imparo_moe_router_pays": [I, I, I, I],
    "imparo_moe_router_blocks": [I],
    # x, w, bias, correction, choice, weight, counts, n_tokens, n_router, k, top, scoring, normalize, scale, always, n_experts,
    # tile_rows, slot_of_entry, entry_of_slot, tiles, max_tiles, stream
    "imparo_moe_router_plan": [P, P, P, P, P, P, P, I, I, I, I, I, I, F, I, I, I, P, P, P, I, P],
    # x, y, h, h_dtype, choice, weight, slot_of_entry, top, n_experts, n_rows_x, rows, w_post, eps_post, w_next, eps_next,
    # out, out_dtype, n_out, width, stream
    "imparo_post_norm_add_moe": [P, P, P, I, P, P, P, I, I, I, P, P, F, P, F, P, I, I, I, P],
    "imparo_moe_tile_rows": [I, I, I],
    "imparo_moe_max_tiles": [I, I, I],
    "imparo_moe_plan": [P, I, I, I, P, P, P, I, P],
    # a, a_ld, gather_div, entry_of_slot, w, out, out_dtype, dtype, tiles, max_tiles, tile_rows, n, k, epilogue, limits, alpha,
    # entry_weight, n_entries, stream
    "imparo_moe_gemm": [P, I, I, P, P, P, I, I, P, I, I, I, I, I, P, F, P, I, P],
    "imparo_moe_combine": [P, P, I, P, P, P, P, I, I, I, I, P],
    # x, delta, n_delta, n_rows_x, rows, w_post, eps_post, w_next, eps_next, out, out_dtype, n_out, width, stream
    "imparo_post_norm_add": [P, P, I, I, P, P, F, P, F, P, I, I, I, P],
    "imparo_rows_parts": [I],
    # x, ssq_in, n_parts, eps, w, bias, y, out_dtype, x_io, ssq_out, weighted_out, weighted_by, m, n, k, epilogue, stream
    "imparo_rows_gemm_conv": [P, P, P, P, P, P, I, I, I, I, I, P],
    "imparo_rows_gemm_tanh": [P, P, P, P, P, F, P, P, I, I, I, P],
    "imparo_rows_gemm": [P, P, I, F, P, P, P, I, P, P, P, P, I, I, I, I, P],
    "imparo_in_proj_conv_decode_normed": [P, P, I, F, P, P, P, P, P, P, P, I, I, I, I, I, I, P],
    "imparo_rows_fold_pays": [I, I, I],
    # a model's step as one call (kernels/program.py holds the structures)
    "imparo_program_new": ([I, I], P),
    "imparo_program_delete": ([P], None),
    "imparo_program_set_fold": [P, I],
    "imparo_program_embedding": [P, P, I, I, I],
    "imparo_program_norm": [P, P, F, I, I],
    "imparo_program_attention": [P, P],
    "imparo_program_short_conv": [P, P],
    "imparo_program_swiglu": [P, P],
    "imparo_program_head": [P, P, F, I, P],
    "imparo_program_n_regions": [P],
    "imparo_program_region_name": ([P, I], ctypes.c_char_p),
    "imparo_program_bind": [P, I, P, c_int64],
    "imparo_program_needs": [P, P, P],
    "imparo_program_needs_up_to": [P, P, P],
    "imparo_program_run": [P, P, P, P],
    "imparo_program_error": ([P], ctypes.c_char_p),
}


class KernelLibraryError(RuntimeError):
    pass


def library() -> ctypes.CDLL:
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        path = _build.library_path()
        if not os.path.isfile(path):
            path = _rebuild("is not built")
        try:
            lib = ctypes.CDLL(path)
        except OSError as e:
            raise KernelLibraryError(f"cannot load {path}: {e}") from e
        built_from = _hash_in(lib, "imparo_hip_source_hash")
        if built_from != _build.source_hash():
            # older than its sources (or from before libraries carried a hash): never used silently
            import _ctypes
            _ctypes.dlclose(lib._handle)
            path = _rebuild(f"at {path} was built from other sources ({built_from}) than those beside it")
            lib = ctypes.CDLL(path)
            if _hash_in(lib, "imparo_hip_source_hash") != _build.source_hash():
                raise KernelLibraryError(f"{path} still does not match its sources after a rebuild")
        for name, argtypes in _SIGNATURES.items():
            try:
                fn = getattr(lib, name)
            except AttributeError:
                raise KernelLibraryError(f"{path} lacks the entry point {name}; rebuild it "
                                         f"(python -m imparo_amd.csrc.build)") from None
            if isinstance(argtypes, tuple):          # (arguments, what it returns) where that is no status
                fn.argtypes, fn.restype = argtypes
            else:
                fn.argtypes, fn.restype = argtypes, c_int
        _lib = lib
        return _lib


def _hash_in(lib: ctypes.CDLL, name: str) -> str:
    try:
        fn = getattr(lib, name)
    except AttributeError:
        return "none"
    fn.restype = ctypes.c_char_p
    fn.argtypes = []
    return fn().decode("ascii", "replace")


def _rebuild(why: str) -> str:
    try:
        return _build.build(verbose=True)
    except Exception as e:  # no silent fallback: say why there is no library
        raise KernelLibraryError(f"the gfx950 kernel library {why} and building it failed: {e}") from e


def loaded_path() -> str:
    library()
    return _build.library_path()
