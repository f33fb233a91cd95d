"""ctypes binding of libexo_mi355x.so (the C ABI declared in include/exo_mi355x.h).

The library is the only compute path: if it is missing, loading raises and every
operator of this package fails loudly.  There is no CPU or eager-PyTorch fallback.
"""

from __future__ import annotations

import ctypes as C
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "libexo_mi355x.so"

_vp = C.c_void_p
_i = C.c_int
_i64 = C.c_int64
_f = C.c_float


class MoeRows(C.Structure):
    """struct exo_moe_rows: the experts of a decode step."""

    _fields_ = [(n, _vp) for n in ("x", "gate", "up", "down", "shared_gate", "shared_up", "shared_down", "act",
                                   "shared_act", "out", "x_res", "idx", "wt", "logits", "correction")] + \
               [(n, _i) for n in ("rows", "top", "experts", "ff", "shared_ff", "H", "ldx", "lda", "ldsa", "ldl",
                                  "gate_col", "outputs", "renorm", "dtype")] + \
               [(n, _f) for n in ("router_scale", "limit", "alpha", "shift", "shared_limit", "shared_alpha", "shared_shift")]


class Linear(C.Structure):
    """struct exo_linear: a product (or gated pair) with an unquantised matrix."""

    _fields_ = [(n, _vp) for n in ("x", "w", "w_up", "bias", "y", "y2", "mul", "mul_rows")] + \
               [(n, _i) for n in ("M", "N", "n1", "ldx", "ldw", "ldy", "ldy2", "y_f32", "dtype", "act", "ldmul")] + \
               [(n, _f) for n in ("limit", "alpha", "shift", "cubic", "cap")]


class PostNorm(C.Structure):
    """struct exo_post_norm: a sublayer's output on its way into the residual."""

    _fields_ = [(n, _vp) for n in ("x", "branch", "branch2", "gain_a", "gain_b", "gain", "pre", "x_out", "operand")] + \
               [(n, _i) for n in ("H", "ldb", "sum", "center")] + [(n, _f) for n in ("eps", "mult", "keep")]


class PagedAttn(C.Structure):
    """struct exo_paged_attn: one attention layer over a paged pool."""

    _fields_ = [(n, _vp) for n in ("qkv", "k_pool", "v_pool", "table", "slot", "pos", "list", "slopes", "q_gain", "k_gain",
                                   "gate", "freq", "v_mix", "out_gate", "weight_bias", "mean_k", "mean_v", "mean_table",
                                   "conv_w", "ring", "map", "q_out", "out")] + \
               [(n, _f) for n in ("scale", "eps", "softcap", "mix", "rot_amp")] + \
               [(n, _i) for n in ("n", "heads", "kv_heads", "dim", "vdim", "ldq", "ldk", "ldv", "ldo", "ldg", "max_pages",
                                  "window", "keep_first", "unit_qk", "whole_norm", "rot", "ldmix", "prepared", "dtype",
                                  "ldog", "mean_pages", "pool", "plus_one", "rot_half", "taps", "ldqo", "shared_kv")]


class LatentAttn(C.Structure):
    """struct exo_latent_attn: one latent-attention layer over a paged pool."""

    _fields_ = [(n, _vp) for n in ("q", "q_latent", "kv", "gain", "freq", "pool", "table", "slot", "pos", "list", "out",
                                   "parts")] + \
               [("parts_floats", _i64), ("scale", _f), ("eps", _f)] + \
               [(n, _i) for n in ("n", "heads", "rank", "rot", "rot_col", "ldq", "ldql", "ldkv", "ldk", "ldo", "max_pages",
                                  "prepared", "nsplit", "dtype")]


class HeadLinear(C.Structure):
    """struct exo_head_linear_args: a product with a matrix per head."""

    _fields_ = [("x", _vp), ("w", _vp), ("parts", _vp), ("parts_floats", _i64), ("y", _vp), ("list", _vp)] + \
               [(n, _i) for n in ("n", "heads", "N", "K", "ldx", "x_head", "ldw", "ldy", "y_head", "nsplit", "dtype")]


class LatentPrompt(C.Structure):
    """struct exo_latent_prompt_args: portions of prompts over expanded keys and values."""

    _fields_ = [(n, _vp) for n in ("q", "k", "k_rot", "v", "list", "out")] + [("scale", _f)] + \
               [(n, _i) for n in ("n", "heads", "vdim", "d8", "r8", "ldq", "q_head", "rot_col", "ldk", "ldv", "ldo")]


class Recurrence(C.Structure):
    """struct exo_recurrence: one recurrent mixer."""

    _fields_ = [(n, _vp) for n in (
        "q", "k", "v", "low", "decay_w", "decay_b", "dt_raw", "dt_bias", "decay_rate", "skip", "gate_i", "gate_f", "raw",
        "conv_w", "conv_b", "ring", "act", "cum", "dt", "state", "y", "peak", "peaks", "map", "slot", "pos", "list", "chunks", "seqs")] + \
        [(n, _i) for n in (
            "ldq", "ldk", "ldv", "ldlow", "rank", "lddt", "ldraw", "channels", "taps", "ldact", "ldcum", "lds", "ldy",
            "ldgate", "ldpeaks", "q_channel", "k_channel", "v_channel", "heads", "groups", "dim", "vdim", "per_channel", "n", "n_chunks",
            "n_seqs", "qk_vec", "v_vec", "dtype")] + [("q_scale", _f), ("inv_tau", _f), ("gate_cap", _f)]


class GatedNorm(C.Structure):
    """struct exo_gated_norm: RMS norm of parts of a row with a gate."""

    _fields_ = [(n, _vp) for n in ("y", "gate", "gain", "out", "peaks")] + \
               [(n, _i) for n in ("width", "groups", "period", "ldy", "ldg", "ldo", "gate_first", "dtype", "ldpart", "ldpeaks",
                                  "den", "sigmoid")] + [("eps", _f)]


# name -> (restype, argtypes); mirrors include/exo_mi355x.h one to one
SIGNATURES: dict[str, tuple] = {
    "exo_abi_version": (_i, []),
    "exo_last_error": (C.c_char_p, []),
    "exo_last_variant": (C.c_char_p, []),
    "exo_dequant_two_roundings": (_i, []),
    "exo_unpack_codes": (_i, [_vp, _vp, _i64, _i, _vp]),
    "exo_dequantize": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _vp]),
    "exo_embed_dequant": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_qmv": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_qmv_swiglu": (_i, [_vp] * 8 + [_i, _i, _i, _i, _i, _vp]),
    "exo_norm_qmv": (_i, [_vp, _vp, _f, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_qmv_workspace": (_i64, [_i]),
    "exo_norm_qmv_ws": (_i, [_vp, _vp, _f, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "exo_norm_qmv_swiglu": (_i, [_vp, _vp, _f] + [_vp] * 7 + [_i, _i, _i, _i, _i, _vp]),
    "exo_norm_qmv_swiglu_ws": (_i, [_vp, _vp, _f] + [_vp] * 8 + [_i64, _i, _i, _i, _i, _i, _vp]),
    "exo_moe_group_workspace": (_i64, [_i, _i, _i]),
    "exo_moe_group": (_i, [_vp, _i, _i, _i, _vp, _i64, _vp]),
    "exo_gather_qmm": (_i, [_vp] * 6 + [_i] * 8 + [_vp]),
    "exo_gather_qmm_swiglu": (_i, [_vp] * 9 + [_i] * 8 + [_vp]),
    "exo_qmm": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_qmm_workspace": (_i64, [_i, _i]),
    "exo_qmm_ws": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "exo_qmm_swiglu": (_i, [_vp] * 8 + [_i, _i, _i, _i, _i, _vp]),
    "exo_qmm_swiglu_workspace": (_i64, [_i, _i]),
    "exo_qmm_swiglu_ws": (_i, [_vp] * 9 + [_i64, _i, _i, _i, _i, _i, _vp]),
    "exo_gather_qmv": (_i, [_vp] * 6 + [_i] * 8 + [_vp]),
    "exo_gather_qmv_combine": (_i, [_vp] * 9 + [_i] * 7 + [_vp]),
    "exo_gather_qmv_swiglu": (_i, [_vp] * 9 + [_i] * 7 + [_vp]),
    "exo_norm_gather_qmv_swiglu": (_i, [_vp, _vp, _f] + [_vp] * 8 + [_i] * 7 + [_vp]),
    "exo_norm_route_gather_qmv_swiglu": (_i, [_vp, _vp, _f, _vp, _i] + [_vp] * 9 + [_i] * 7 + [_vp]),
    "exo_add_rmsnorm": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _f, _vp]),
    "exo_rope_kv_append": (_i, [_vp] * 8 + [_f] + [_i] * 6 + [_vp]),
    "exo_rope_kv_append_tab": (_i, [_vp] * 7 + [_i] + [_vp] * 2 + [_f] + [_i] * 6 + [_vp]),
    "exo_sdpa_decode_workspace": (_i64, [_i, _i, _i]),
    "exo_sdpa_decode": (_i, [_vp] * 6 + [_f] + [_i] * 5 + [_vp]),
    "exo_sdpa_decode_static": (_i, [_vp] * 5 + [_f] + [_i] * 5 + [_vp]),
    "exo_attn_decode": (_i, [_vp] * 8 + [_f, _vp, _vp, _f] + [_i] * 5 + [_vp]),
    "exo_attn_decode_hint": (_i, [_vp] * 8 + [_f, _vp, _vp, _f] + [_i] * 6 + [_vp]),
    "exo_rope_table": (_i, [_vp, _vp, _i, _i, _vp]),
    "exo_sdpa_prefill": (_i, [_vp] * 5 + [_f] + [_i] * 6 + [_vp]),
    "exo_kv_export_nhd": (_i, [_vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_kv_import_nhd": (_i, [_vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "exo_swiglu": (_i, [_vp, _vp, _vp, _i64, _vp]),
    "exo_router_topk": (_i, [_vp, _vp, _vp, _i, _i, _i, _i, _vp]),
    "exo_moe_combine": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _vp]),
    "exo_put_i32": (_i, [_vp, _vp, _i, _vp]),
    "exo_argmax_workspace": (_i64, [_i]),
    "exo_argmax_logsumexp": (_i, [_vp] * 6 + [_i, _i, _vp]),
    "exo_embed_rows": (_i, [_vp] * 4 + [_i] * 5 + [_f, _i, _vp]),
    "exo_norm_rows": (_i, [_vp] * 4 + [_i] * 4 + [_f, _i, _i, _vp]),
    "exo_post_norm_add": (_i, [C.POINTER(PostNorm), _i, _i, _i, _vp]),
    "exo_moe_sum_post_norm": (_i, [_vp] * 5 + [_i] * 6 + [C.POINTER(PostNorm), _i, _i, _i, _vp]),
    "exo_moe_route": (_i, [_vp] * 4 + [_i] * 4 + [_f, _i, _vp]),
    "exo_linear_rows": (_i, [C.POINTER(Linear), C.POINTER(Linear), _vp]),
    "exo_linear_pair_workspace": (_i64, [C.POINTER(Linear)]),
    "exo_linear_gemm": (_i, [C.POINTER(Linear), _vp, _i64, _vp]),
    "exo_post_linear_fits": (_i, [_i] * 5),
    "exo_post_linear": (_i, [C.POINTER(PostNorm), C.POINTER(Linear), _vp]),
    "exo_dense_grouped_gemm": (_i, [_vp] * 5 + [_f] * 3 + [_i] * 9 + [_vp]),
    "exo_moe_glu_rows": (_i, [C.POINTER(MoeRows), _vp]),
    "exo_moe_down_rows": (_i, [C.POINTER(MoeRows), _vp]),
    "exo_paged_prepare": (_i, [C.POINTER(PagedAttn), _vp]),
    "exo_paged_means": (_i, [C.POINTER(PagedAttn), _vp]),
    "exo_paged_append": (_i, [C.POINTER(PagedAttn), _vp]),
    "exo_paged_attn_workspace": (_i64, [_i] * 4),
    "exo_paged_attn_rows": (_i, [C.POINTER(PagedAttn), _i, _i, _vp, _i64, _vp]),
    "exo_paged_prompt_block": (_i, [_i, _i]),
    "exo_paged_attn_prompt": (_i, [C.POINTER(PagedAttn), _vp]),
    "exo_latent_prepare": (_i, [C.POINTER(LatentAttn), _vp]),
    "exo_latent_parts": (_i64, [_i] * 4),
    "exo_latent_rows": (_i, [C.POINTER(LatentAttn), _i, _vp]),
    "exo_head_linear": (_i, [C.POINTER(HeadLinear), _vp]),
    "exo_latent_gather": (_i, [C.POINTER(LatentAttn), _vp, _i, _vp, _vp, _vp]),
    "exo_latent_prompt": (_i, [C.POINTER(LatentPrompt), _vp]),
    "exo_recur_chunk": (_i, []),
    "exo_recur_workspace": (_i64, [C.POINTER(Recurrence)]),
    "exo_recur_chunks": (_i, [C.POINTER(Recurrence), _vp, _i64, _vp]),
    "exo_recur_step": (_i, [C.POINTER(Recurrence), _vp]),
    "exo_gated_norm_rows": (_i, [C.POINTER(GatedNorm), _vp, _i, _vp]),
    "exo_sample_workspace": (_i64, [_i]),
    "exo_sample": (_i, [_vp] * 13 + [_i64, _i, _i, _i, _i, _vp]),
}


class NativeError(RuntimeError):
    pass


_lib = None


def load() -> C.CDLL:
    """Load the shared library (once).  Raises NativeError when it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not LIB_PATH.exists():
        raise NativeError(
            f"{LIB_PATH} not found: build it with `python -m exo_amd.build` "
            "(there is no fallback path)"
        )
    lib = C.CDLL(str(LIB_PATH))
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)  # AttributeError if the symbol is not exported
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = load().exo_last_error().decode("utf-8", "replace")
        if rc == -1:
            raise ValueError(f"{what}: {msg}")
        raise NativeError(f"{what}: {msg} (rc={rc})")


def last_variant() -> str:
    """The kernel instance the calling thread's latest matmul / attention call selected."""
    return load().exo_last_variant().decode("utf-8", "replace")
