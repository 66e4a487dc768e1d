"""ctypes binding of libnvx_spec.so (the C ABI declared in include/nvx_spec.h).

torch is imported first so the HIP runtime it bundles (libamdhip64.so.7) is the
one the library binds to; torch provides device memory and streams, every kernel
of the verify path lives in the library.  There is no fallback: if the library is
missing or fails to load, using any op raises.
"""
import ctypes
from ctypes import c_void_p, c_int32, c_int64, c_float, c_size_t, c_double, POINTER
from pathlib import Path

import torch  # noqa: F401  (loads the HIP runtime before the library)

LIB_PATH = Path(__file__).resolve().parent / "_lib" / "libnvx_spec.so"

DTYPE_F32, DTYPE_BF16, DTYPE_F16 = 0, 1, 2
TIMER_NGRAM, TIMER_STORE_KV, TIMER_KV_COMPACT, TIMER_TREE_ATTENTION, TIMER_SOFTMAX, \
    TIMER_REJECTION, TIMER_TOPK = range(7)


class DecoderLayerArgs(ctypes.Structure):
    """nvx_decoder_layer_args"""
    _fields_ = ([(n, c_void_p) for n in (
        "hidden", "residual", "residual_in_out", "residual_out", "out", "input_norm", "qkv_weight",
        "q_norm", "k_norm", "o_weight", "post_norm", "gate_up_weight", "down_weight", "positions",
        "cos_sin_cache", "k_cache", "v_cache", "slot_mapping", "block_tables", "cu_seqlens_q",
        "context_lens", "tree_mask")]
        + [("cache_positions", c_int64)]
        + [(n, c_int32) for n in (
            "num_tokens", "hidden_size", "inter_size", "num_heads", "num_kv_heads", "head_dim",
            "num_seqs", "max_seqlen_q", "max_context_len", "block_size", "block_table_stride")]
        + [(n, c_float) for n in ("input_eps", "qk_eps", "post_eps", "scale")])


_SIGS = {
    "nvx_version": ([], c_int32),
    "nvx_last_error": ([], ctypes.c_char_p),
    "nvx_ngram_propose": ([c_void_p, c_void_p, c_int32, c_int32, c_int32, c_int32, c_void_p,
                           c_void_p, c_void_p], c_int32),
    "nvx_store_kvcache": ([c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_void_p,
                           c_int32, c_int32, c_void_p], c_int32),
    "nvx_kv_compact": ([c_void_p, c_void_p, c_int64, c_int32, c_int32, c_int32, c_void_p, c_int32,
                        c_void_p, c_void_p, c_int32, c_void_p, c_int32, c_void_p], c_int32),
    "nvx_tree_attention_workspace_size": ([c_int32] * 7, c_size_t),
    "nvx_tree_attention": ([c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int32, c_void_p,
                            c_void_p, c_void_p, c_int32, c_int32, c_int32, c_int32, c_int32,
                            c_int32, c_int32, c_int32, c_float, c_void_p, c_size_t, c_void_p],
                           c_int32),
    "nvx_tree_attention_noalloc_scratch_bytes": ([], c_size_t),
    "nvx_tree_attention_noalloc": ([c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int32,
                                    c_void_p, c_void_p, c_void_p, c_int32, c_int32, c_int32,
                                    c_int32, c_int32, c_int32, c_int32, c_int32, c_float,
                                    c_void_p], c_int32),
    "nvx_temperature_softmax": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_int32, c_int32,
                                 c_void_p], c_int32),
    "nvx_sample": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_void_p, c_int32, c_int32,
                    c_void_p], c_int32),
    "nvx_rejection_sample_tree": ([c_void_p, c_int64, c_void_p, c_int64, c_int32, c_void_p,
                                   c_void_p, c_void_p, c_int32, c_void_p, c_void_p, c_void_p,
                                   c_int32, c_int32, c_void_p, c_void_p, c_void_p, c_void_p,
                                   c_void_p, c_size_t, c_void_p], c_int32),
    "nvx_rejection_sample_chain": ([c_void_p, c_int64, c_void_p, c_int64, c_int32, c_void_p, c_int32,
                                    c_int32, c_void_p, c_void_p, c_void_p, c_int32, c_void_p,
                                    c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p],
                                   c_int32),
    "nvx_rejection_walk_workspace_size": ([c_int32], c_size_t),
    "nvx_rmsnorm": ([c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p, c_int32, c_int32,
                     c_float, c_void_p], c_int32),
    "nvx_qk_norm_rope": ([c_void_p, c_int64, c_int32, c_int32, c_int32, c_void_p, c_void_p,
                          c_void_p, c_void_p, c_int64, c_int32, c_void_p, c_void_p, c_void_p,
                          c_void_p, c_void_p, c_float, c_void_p], c_int32),
    "nvx_silu_mul": ([c_void_p, c_int64, c_void_p, c_int32, c_int32, c_void_p], c_int32),
    "nvx_skinny_gemm": ([c_void_p, c_int64, c_void_p, c_void_p, c_int32, c_int32, c_int32, c_int32,
                         c_void_p], c_int32),
    "nvx_decoder_layer_scratch_size": ([POINTER(DecoderLayerArgs)], c_size_t),
    "nvx_decoder_layer": ([POINTER(DecoderLayerArgs), c_void_p, c_size_t, c_void_p], c_int32),
    "nvx_softmax_stats": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_int32, c_int32,
                           c_void_p], c_int32),
    "nvx_softmax_from_stats": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_void_p, c_int32,
                                c_int32, c_void_p], c_int32),
    "nvx_rejection_sample_tree_logits": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_void_p,
                                          c_int64, c_int32, c_void_p, c_void_p, c_void_p, c_int32,
                                          c_void_p, c_void_p, c_void_p, c_int32, c_int32, c_void_p,
                                          c_void_p, c_void_p, c_void_p, c_void_p, c_size_t,
                                          c_void_p], c_int32),
    "nvx_rejection_sample_tree_logits_lazy": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p,
                                               c_void_p, c_int64, c_int32, c_void_p, c_void_p,
                                               c_void_p, c_int32, c_void_p, c_void_p, c_void_p,
                                               c_int32, c_int32, c_void_p, c_void_p, c_void_p,
                                               c_void_p, c_void_p, c_size_t, c_void_p], c_int32),
    "nvx_rejection_verify_logits": ([c_void_p, c_int32, c_int64, c_void_p, c_void_p, c_void_p, c_int64,
                                     c_int32, c_void_p, c_void_p, c_void_p, c_int32, c_void_p,
                                     c_void_p, c_int32, c_int32, c_void_p, c_void_p, c_void_p,
                                     c_void_p, c_void_p, c_size_t, c_void_p], c_int32),
    "nvx_topk_logprobs": ([c_void_p, c_int32, c_int64, c_int32, c_int32, c_int32, c_void_p,
                           c_void_p, c_void_p], c_int32),
    "nvx_topk_logprobs_i64": ([c_void_p, c_int32, c_int64, c_int32, c_int32, c_int32, c_void_p,
                               c_void_p, c_void_p], c_int32),
    "nvx_rejection_walk_max_width": ([c_int32], c_int32),
    "nvx_timing_enable": ([c_int32], c_int32),
    "nvx_timing_read": ([c_int32, POINTER(c_double), POINTER(c_int64)], c_int32),
    "nvx_timing_reset": ([], c_int32),
}

EXPORTED = tuple(_SIGS)

_lib = None


def lib():
    """Load (once) and return the library; raises if it is not built."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise ImportError(
                f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; "
                f"g.build()'` (hipcc, gfx950). The verify path has no CPU fallback.")
        handle = ctypes.CDLL(str(LIB_PATH))
        for name, (args, res) in _SIGS.items():
            fn = getattr(handle, name)
            fn.argtypes = args
            fn.restype = res
        _lib = handle
    return _lib


def check(rc):
    if rc != 0:
        msg = lib().nvx_last_error().decode(errors="replace")
        raise RuntimeError(f"libnvx_spec: {msg} (code {rc})")


def ptr(t):
    """Device pointer of a tensor (None -> NULL), as the int a c_void_p argument takes."""
    return None if t is None else t.data_ptr()


def stream_of(t):
    """Handle of the current stream of the tensor's device, without a Stream object."""
    return torch._C._cuda_getCurrentRawStream(t.get_device())


def require_cuda(*tensors):
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("libnvx_spec ops run on the GPU only: got a tensor on "
                               f"{t.device}")


def timing_enable(on=True):
    check(lib().nvx_timing_enable(1 if on else 0))


def timing_reset():
    check(lib().nvx_timing_reset())


def timing_read(kernel_id):
    ms, n = c_double(0), c_int64(0)
    check(lib().nvx_timing_read(kernel_id, ctypes.byref(ms), ctypes.byref(n)))
    return ms.value, n.value
