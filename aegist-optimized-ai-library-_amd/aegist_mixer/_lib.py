"""ctypes loader for libaegist_mixer.so: one declaration per exported symbol of
include/aegist_mixer.h, and a checked-call helper that raises on a non-zero return.

The library is the only compute path: if it is missing or fails to load, importing the ops
raises — there is no CPU fallback."""
from __future__ import annotations

import ctypes as C
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "libaegist_mixer.so"

F32, BF16, I8 = 0, 1, 2

P = C.c_void_p
I = C.c_int
F = C.c_float
LL = C.c_longlong
SZ = C.c_size_t

# name -> (restype, argtypes); mirrors include/aegist_mixer.h
SIGNATURES: dict[str, tuple] = {
    "aegist_last_error": (C.c_char_p, []),
    "aegist_version": (C.c_char_p, []),
    "aegist_set_device": (I, [I]),
    "aegist_bind_workspace": (I, [P, SZ]),
    "aegist_malloc": (I, [C.POINTER(C.c_void_p), SZ]),
    "aegist_free": (I, [P]),
    "aegist_memcpy_htod": (I, [P, P, SZ, P]),
    "aegist_memcpy_dtoh": (I, [P, P, SZ, P]),
    "aegist_memcpy_dtod": (I, [P, P, SZ, P]),
    "aegist_memset": (I, [P, I, SZ, P]),
    "aegist_mem_info": (I, [C.POINTER(SZ), C.POINTER(SZ)]),
    "aegist_stream_sync": (I, [P]),
    "aegist_fill_normal": (I, [P, SZ, I, C.c_uint64, F, F, P]),
    "aegist_znorm": (I, [P, P, P, I, I, F, P]),
    "aegist_attn_prep": (I, [P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, F, F, P]),
    "aegist_attention_gated": (I, [P, P, P, P, P, I, I, I, I, I, F, P]),
    "aegist_attention_gated_workspace_bytes": (SZ, [I, I, I, I]),
    "aegist_attention_gated_ws": (I, [P, P, P, P, P, I, I, I, I, I, F, P, SZ, P]),
    "aegist_delta_gates": (I, [P, P, P, P, P, P, I, I, I, P]),
    "aegist_conv_silu": (I, [P, P, P, P, I, I, P]),
    "aegist_l2norm_heads": (I, [P, I, I, I, I, F, F, P]),
    "aegist_delta_scan": (I, [P, P, P, P, I, I, I, I, P]),
    "aegist_delta_scan_workspace_bytes": (SZ, [I, I, I]),
    "aegist_delta_scan_ws": (I, [P, P, P, P, I, I, I, I, P, SZ, P]),
    "aegist_gated_norm": (I, [P, P, P, P, I, I, I, F, P]),
    "aegist_delta_decode_step": (I, [P, I, P, P, P, P, P, P, I, I, I, I, F, F, P]),
    "aegist_delta_recurrent": (I, [P, P, P, I, LL, LL, LL, LL, LL, LL, P, P, P, P, I, LL, LL, LL,
                                   I, I, I, I, I, F, F, P]),
    "aegist_delta_chunked_workspace_bytes": (SZ, [I, I, I]),
    "aegist_delta_chunked": (I, [P, P, P, I, LL, LL, LL, LL, LL, LL, P, P, P, P, I, LL, LL, LL,
                                 I, I, I, I, I, F, F, P, SZ, P]),
    "aegist_rope_inv_freq": (I, [P, I, F]),
    "aegist_attention_decode_workspace_bytes": (SZ, [I, I, I, I]),
    "aegist_attention_decode": (I, [P, P, P, I, P, P, P, P, P, I, I, I, I, I, I, I, I, F, F, P, SZ, P]),
    "aegist_attention_decode_noalloc": (I, [P, P, P, I, P, P, P, P, P, I, I, I, I, I, I, I, I, F, F, P]),
    "aegist_attention_core": (I, [P, P, P, P, P, I, I, I, I, I, I, F, P, SZ, P]),
    "aegist_attention_core_workspace_bytes": (SZ, [I, I, I, I, I]),
    "aegist_stack_create": (I, [P, C.POINTER(C.c_void_p)]),
    "aegist_stack_destroy": (I, [P]),
    "aegist_stack_set_layer": (I, [P, I, P]),
    "aegist_stack_reset": (I, [P, P]),
    "aegist_stack_length": (I, [P]),
    "aegist_stack_forward": (I, [P, P, I, I, P]),
    "aegist_embed_bf16": (I, [P, P, P, I, I, P]),
    "aegist_stack_snapshot": (I, [P, P]),
    "aegist_stack_crop": (I, [P, I, P]),
    "aegist_stack_state_bytes": (SZ, [P, I]),
    "aegist_stack_save_state": (I, [P, I, P, SZ, P]),
    "aegist_stack_load_state": (I, [P, I, I, P, SZ, P]),
    "aegist_idx_prep": (I, [P, P, P, P, I, I, I, I, I, F, F, P]),
    "aegist_idx_blocks": (I, [P, P, P, I, I, I, I, I, F, F, P]),
    "aegist_idx_scores": (I, [P, P, P, I, I, I, I, I, I, P]),
    "aegist_idx_select": (I, [P, P, P, I, I, I, I, I, P]),
    "aegist_idx_select_workspace_bytes": (SZ, [I, I, I, I]),
    "aegist_idx_select_ws": (I, [P, P, P, I, I, I, I, I, P, SZ, P]),
    "aegist_attention_gated_list": (I, [P, P, P, P, P, I, I, I, I, I, F, P, P, I, I, P]),
    "aegist_attention_gated_list_workspace_bytes": (SZ, [I, I, I, I, I, I]),
    "aegist_attention_gated_list_ws": (I, [P, P, P, P, P, I, I, I, I, I, F, P, P, I, I, P, SZ, P]),
    "aegist_gated_norm2": (I, [P, P, P, P, I, I, I, F, I, P]),
    "aegist_gemv_i8": (I, [P, P, P, P, I, I, I, P]),
    "aegist_gemv_bf16": (I, [P, P, P, I, I, P]),
    "aegist_gemm_i8": (I, [P, P, P, P, I, I, I, I, P]),
    "aegist_linear": (I, [P, I, LL, P, I, P, P, LL, I, I, I, I, P]),
    "aegist_linear_multi": (I, [P, I, LL, I, I, P, P, P, P, P, I, I, I, P]),
    "aegist_router_topk": (I, [P, P, P, P, I, I, I, I, P]),
    "aegist_router_topk_workspace_bytes": (SZ, [I, I]),
    "aegist_router_topk_ws": (I, [P, P, P, P, I, I, I, I, P, SZ, P]),
    "aegist_moe_workspace_bytes": (SZ, [I, I, I, I, I]),
    "aegist_moe_experts": (I, [P, P, P, P, P, I, I, I, I, I, P, P, P, SZ, P]),
    "aegist_shared_gate_add": (I, [P, P, P, P, I, I, P]),
    "aegist_silu_mul": (I, [P, P, P, LL, P]),
}


MAX_LAYERS = 64


class StackConfig(C.Structure):
    """AegistStackConfig of include/aegist_mixer.h."""
    _fields_ = [("n_layers", I), ("d_model", I), ("hk", I), ("hv", I), ("n_heads", I), ("n_kv", I),
                ("head_dim", I), ("rotary_dim", I), ("rope_theta", F), ("eps", F), ("max_batch", I),
                ("max_tokens", I), ("max_context", I), ("layer_is_attn", C.c_ubyte * MAX_LAYERS)]


class LayerWeights(C.Structure):
    """AegistLayerWeights of include/aegist_mixer.h (device pointers)."""
    _fields_ = [(name, P) for name in ("norm1", "w_qkv", "w_z", "w_b", "w_a", "conv_w", "a_log", "dt_bias",
                                       "gnorm_w", "w_out", "w_q", "w_k", "w_v", "w_o", "q_norm", "k_norm")]


class AegistError(RuntimeError):
    """A non-zero return code from libaegist_mixer; the message is aegist_last_error()."""

    def __init__(self, fn: str, code: int, msg: str):
        super().__init__(f"{fn} failed ({code}): {msg}")
        self.code = code


_lib = None


def lib():
    """Load the library once and bind every declared symbol (missing symbols raise)."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise ImportError(f"{LIB_PATH} is missing: build it with "
                              f"`python aegist-optimized-ai-library-_amd/build.py` (no CPU fallback exists)")
        L = C.CDLL(str(LIB_PATH))
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name, None)
            if fn is None:
                continue  # reported by call() if used; the export test checks completeness
            fn.restype = res
            fn.argtypes = args
        _lib = L
    return _lib


_fns: dict = {}  # bound entry points by name (an attribute lookup per call costs about a microsecond)


def call(name: str, *args) -> None:
    fn = _fns.get(name)
    if fn is None:
        fn = getattr(lib(), name, None)
        if fn is None:
            raise AegistError(name, -99, "symbol not exported by this build of libaegist_mixer.so")
        _fns[name] = fn
    rc = fn(*args)
    if rc != 0:
        raise AegistError(name, rc, lib().aegist_last_error().decode(errors="replace"))


def last_error() -> str:
    return lib().aegist_last_error().decode(errors="replace")
