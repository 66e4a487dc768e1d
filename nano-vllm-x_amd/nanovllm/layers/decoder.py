"""A decoder layer's step over few rows as one library call (``nvx_decoder_layer``).

``few_rows_layer`` serves ``Qwen3DecoderLayer.forward`` (reference
nanovllm/models/qwen3.py:140-160) when a step brings at most ``MAX_ROWS`` rows and every
module of the layer is the plain one; otherwise it returns None and the layer runs
module by module.
"""
import ctypes

import torch
from torch import nn
from torch.nn.modules import module as _module

from .. import _C
from ..utils.context import get_context
from .activation import SiluAndMul
from .attention import Attention
from .layernorm import RMSNorm

MAX_ROWS = 32

# Up to 16 rows the call takes less GPU time than the modules at every size measured
# (hidden 1024 to 5120 replayed as graphs, weights from HBM: 0.46 to 0.91 of the modules'
# time, though single projections of 9 to 16 rows can be slower than hipBLASLt's), and it
# saves launches.  At 17 to 32 rows re-reading x for every tile of the weights costs more
# than that once the weights are large: us per layer of 32 rows, call and modules,
# hidden 1024 58, 77; 2048 81, 88 (intermediate 8192: 93, 91); 2560 122, 106; 3072 110, 99;
# 4096 150, 140.
ROWS_ANY, HIDDEN_ALL_ROWS = 16, 2048


def _plain(m, kind):
    """m is exactly a `kind`, and calling it runs that class's forward and nothing else."""
    d = m.__dict__
    return type(m) is kind and not (d["_forward_hooks"] or d["_forward_pre_hooks"]) \
        and "forward" not in d


def _weight(m, kind, shape, dev):
    """The weight of a plain, bias-free module, or None if it is not what the kernels read."""
    if not _plain(m, kind):
        return None
    p = m.__dict__["_parameters"]
    w = p.get("weight")
    if type(w) is not nn.Parameter or p.get("bias") is not None:
        return None
    if w.dtype is not torch.bfloat16 or w.shape != shape or w.get_device() != dev \
            or not w.is_contiguous():
        return None
    w = w.data_ptr()
    return w if w % 16 == 0 else None


def _bf16(t, dev, shape=None):
    return (t.dtype is torch.bfloat16 and t.get_device() == dev and t.is_contiguous()
            and (shape is None or t.shape == shape) and t.data_ptr() % 16 == 0)


def _i32(t, dev):
    return t is not None and t.dtype is torch.int32 and t.get_device() == dev and t.is_contiguous()


def few_rows_layer(layer, attention_type, mlp_type, positions, hidden, residual, aux=None):
    """(out, residual) of the layer, or None where the modules have to run one by one:
    more rows, gradients, hooks, replaced modules, other dtypes, layouts or contexts
    (whose errors the modules raise)."""
    if hidden.dim() != 2 or not 0 < hidden.shape[0] <= MAX_ROWS or not hidden.is_cuda \
            or (hidden.shape[0] > ROWS_ANY and hidden.shape[1] > HIDDEN_ALL_ROWS) or torch.is_grad_enabled() \
            or torch.is_autocast_enabled() \
            or _module._global_forward_hooks or _module._global_forward_pre_hooks:
        return None
    ctx = get_context()
    shape = hidden.shape
    N, H = shape
    dev = hidden.get_device()
    mods = layer.__dict__["_modules"]
    sa, mlp, norm_in, norm_post = (mods["self_attn"], mods["mlp"], mods["input_layernorm"],
                                   mods["post_attention_layernorm"])
    if not (_plain(sa, attention_type) and _plain(mlp, mlp_type)):
        return None  # replaced modules need not have the submodules read below
    am, mm = sa.__dict__["_modules"], mlp.__dict__["_modules"]
    attn, rope = am["attn"], am["rotary_emb"]
    if not (_plain(attn, Attention) and _plain(mm["act_fn"], SiluAndMul)):
        return None
    Hq, Hkv, D = sa.num_heads, sa.num_kv_heads, sa.head_dim
    down = mm["down_proj"].__dict__["_parameters"].get("weight")
    if down is None or down.dim() != 2 or H % 64 or down.shape[1] % 64:
        return None
    inter = down.shape[1]
    weights = [_weight(norm_in, RMSNorm, (H,), dev),
               _weight(am["qkv_proj"], nn.Linear, ((Hq + 2 * Hkv) * D, H), dev),
               _weight(am["q_norm"], RMSNorm, (D,), dev) if sa.qk_norm else 0,
               _weight(am["k_norm"], RMSNorm, (D,), dev) if sa.qk_norm else 0,
               _weight(am["o_proj"], nn.Linear, (H, Hq * D), dev),
               _weight(norm_post, RMSNorm, (H,), dev),
               _weight(mm["gate_up_proj"], nn.Linear, (2 * inter, H), dev),
               _weight(mm["down_proj"], nn.Linear, (H, inter), dev)]
    if None in weights:
        return None
    kc, vc = attn.k_cache, attn.v_cache
    slots, bt, cu, lens, mask = (ctx.slot_mapping, ctx.block_tables, ctx.cu_seqlens_q,
                                 ctx.context_lens, ctx.tree_mask)
    max_ctx = ctx.max_seqlen_k if ctx.is_prefill else ctx.max_context_len
    if ctx.is_prefill:
        mask = None
    if not (max_ctx and ctx.max_seqlen_q and kc.dim() == 4 and kc.shape[2:] == (Hkv, D)
            and kc.shape == vc.shape and _bf16(kc, dev) and _bf16(vc, dev) and _bf16(hidden, dev)
            and (residual is None or _bf16(residual, dev, shape))
            and _i32(slots, dev) and slots.numel() == N and _i32(cu, dev) and _i32(lens, dev)
            and _i32(bt, dev) and bt.dim() == 2 and positions.dtype is torch.int64
            and positions.get_device() == dev and positions.is_contiguous()
            and positions.numel() == N and attn.num_kv_heads == Hkv and attn.num_heads == Hq):
        return None
    if mask is not None and (mask.dtype not in (torch.int64, torch.uint64) or mask.numel() != N
                             or not mask.is_contiguous() or mask.get_device() != dev):
        return None
    table = rope.cos_sin_cache
    if not (table.dtype is torch.float32 and table.get_device() == dev):
        return None
    out, res_out = torch.empty_like(hidden), torch.empty_like(hidden)
    mid = None
    if aux is not None:  # the residual stream entering the attention
        mid = hidden if residual is None else torch.empty_like(hidden)
        aux.append(mid)
    args = _C.DecoderLayerArgs(
        hidden.data_ptr(), None if residual is None else residual.data_ptr(),
        None if mid is None else mid.data_ptr(), res_out.data_ptr(), out.data_ptr(), *weights,
        positions.data_ptr(), table.data_ptr(), kc.data_ptr(), vc.data_ptr(), slots.data_ptr(),
        bt.data_ptr(), cu.data_ptr(), lens.data_ptr(), None if mask is None else mask.data_ptr(),
        rope.max_positions, N, H, inter, Hq, Hkv, D, lens.numel(), ctx.max_seqlen_q, max_ctx,
        kc.shape[1], bt.shape[1], norm_in.eps, am["q_norm"].eps if sa.qk_norm else 0.0,
        norm_post.eps, attn.scale)
    L = _C.lib()
    ref = ctypes.byref(args)
    scratch = torch.empty(L.nvx_decoder_layer_scratch_size(ref), dtype=torch.uint8,
                          device=hidden.device)
    _C.check(L.nvx_decoder_layer(ref, scratch.data_ptr(), scratch.numel(), _C.stream_of(hidden)))
    return out, res_out
