"""Qwen3 decoder (single GPU) calling the verify-path attention layer.

Mirrors the reference's nanovllm/models/qwen3.py:14-216 (module names, fused
qkv_proj / gate_up_proj, q/k RMSNorm, NeoX RoPE, add+RMSNorm residual stream,
``compute_logits`` over every row).  Tensor parallelism is left out: one process
drives one GPU.  Dense projections are torch (hipBLASLt) GEMMs; attention,
RMSNorm, q/k-norm + RoPE and SiLU-mul run on the HIP library.  A layer's step over a
few rows is one library call, its projections included (layers/decoder.py).
"""
import torch
from torch import nn

from nanovllm import _C
from nanovllm.layers.activation import SiluAndMul
from nanovllm.layers.attention import Attention
from nanovllm.layers.decoder import few_rows_layer
from nanovllm.layers.layernorm import RMSNorm
from nanovllm.layers.rotary_embedding import get_rope
from nanovllm.utils.context import get_context


class Qwen3Attention(nn.Module):

    def __init__(self, hidden_size, num_heads, num_kv_heads, max_position=4096 * 32,
                 head_dim=None, rms_norm_eps=1e-06, qkv_bias=False, rope_theta=10000,
                 rope_scaling=None, input_size=None, qk_norm=None):
        super().__init__()
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = head_dim or hidden_size // num_heads
        if self.head_dim != 128:
            raise ValueError(f"the fused q/k-norm + RoPE kernel needs head_dim 128 "
                             f"(got {self.head_dim})")
        self.q_size = self.num_heads * self.head_dim
        self.kv_size = self.num_kv_heads * self.head_dim
        self.scaling = self.head_dim ** -0.5
        self.qkv_bias = qkv_bias
        # input_size: width of the attention input (2*hidden in an EAGLE-3 draft layer)
        self.qkv_proj = nn.Linear(input_size or hidden_size, self.q_size + 2 * self.kv_size,
                                  bias=qkv_bias)
        self.o_proj = nn.Linear(self.q_size, hidden_size, bias=False)
        if isinstance(rope_scaling, dict):
            rope_theta = rope_scaling.get("rope_theta", rope_theta)
        self.rotary_emb = get_rope(self.head_dim, self.head_dim, max_position, rope_theta)
        self.attn = Attention(self.num_heads, self.head_dim, self.scaling, self.num_kv_heads)
        # Qwen3 normalises q and k per head when the projection has no bias (reference
        # qwen3.py:50-52); qk_norm=False gives a Llama-style layer (EAGLE-3 heads)
        self.qk_norm = (not qkv_bias) if qk_norm is None else qk_norm
        if self.qk_norm:
            self.q_norm = RMSNorm(self.head_dim, eps=rms_norm_eps)
            self.k_norm = RMSNorm(self.head_dim, eps=rms_norm_eps)

    def forward(self, positions, hidden_states):
        qkv = self.qkv_proj(hidden_states)
        N = qkv.shape[0]
        q = torch.empty(N, self.num_heads, self.head_dim, dtype=qkv.dtype, device=qkv.device)
        slots = get_context().slot_mapping
        k_cache, v_cache = self.attn.k_cache, self.attn.v_cache
        fused_store = slots is not None and k_cache.numel() > 0
        k = None if fused_store else torch.empty(N, self.num_kv_heads, self.head_dim,
                                                 dtype=qkv.dtype, device=qkv.device)
        if fused_store and (k_cache.dtype != qkv.dtype or slots.dtype != torch.int32
                            or slots.numel() != N or k_cache.stride(-3) != self.kv_size):
            raise ValueError("Qwen3Attention: cache / slot_mapping do not match the layer")
        # q/k RMSNorm + RoPE in one pass (reference qwen3.py:82-85), K and V stored
        # into the paged cache by the same kernel (attention.py:62-63)
        _C.require_cuda(qkv, positions)
        rope = self.rotary_emb
        _C.check(_C.lib().nvx_qk_norm_rope(
            _C.ptr(qkv), qkv.stride(0), self.num_heads, self.num_kv_heads, self.head_dim,
            _C.ptr(self.q_norm.weight) if self.qk_norm else None,
            _C.ptr(self.k_norm.weight) if self.qk_norm else None, _C.ptr(positions),
            _C.ptr(rope.cos_sin_cache), rope.max_positions, N, _C.ptr(q), _C.ptr(k),
            _C.ptr(k_cache) if fused_store else None, _C.ptr(v_cache) if fused_store else None,
            _C.ptr(slots) if fused_store else None,
            float(self.q_norm.eps) if self.qk_norm else 0.0, _C.stream_of(qkv)))
        if fused_store:
            o = self.attn(q, None, None)  # K and V are in the cache already
        else:
            v = qkv[:, self.q_size + self.kv_size:].view(-1, self.num_kv_heads, self.head_dim)
            o = self.attn(q, k, v)
        return self.o_proj(o.flatten(1, -1))


class Qwen3MLP(nn.Module):

    def __init__(self, hidden_size, intermediate_size, hidden_act):
        super().__init__()
        assert hidden_act == "silu"
        self.gate_up_proj = nn.Linear(hidden_size, 2 * intermediate_size, bias=False)
        self.down_proj = nn.Linear(intermediate_size, hidden_size, bias=False)
        self.act_fn = SiluAndMul()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_up_proj(x)))


class Qwen3DecoderLayer(nn.Module):

    def __init__(self, config):
        super().__init__()
        self.self_attn = Qwen3Attention(
            hidden_size=config.hidden_size,
            num_heads=config.num_attention_heads,
            num_kv_heads=config.num_key_value_heads,
            max_position=config.max_position_embeddings,
            rms_norm_eps=config.rms_norm_eps,
            qkv_bias=getattr(config, "attention_bias", False),
            head_dim=getattr(config, "head_dim", None),
            rope_theta=getattr(config, "rope_theta", None) or 1000000,
            rope_scaling=getattr(config, "rope_scaling", None),
        )
        self.mlp = Qwen3MLP(config.hidden_size, config.intermediate_size, config.hidden_act)
        self.input_layernorm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)

    def forward(self, positions, hidden_states, residual, aux=None):
        few = few_rows_layer(self, Qwen3Attention, Qwen3MLP, positions, hidden_states, residual, aux)
        if few is not None:
            return few
        if residual is None:
            hidden_states, residual = self.input_layernorm(hidden_states), hidden_states
        else:
            hidden_states, residual = self.input_layernorm(hidden_states, residual)
        if aux is not None:  # the residual stream entering this layer
            aux.append(residual)
        hidden_states = self.self_attn(positions, hidden_states)
        hidden_states, residual = self.post_attention_layernorm(hidden_states, residual)
        return self.mlp(hidden_states), residual


class Qwen3Model(nn.Module):

    def __init__(self, config):
        super().__init__()
        self.embed_tokens = nn.Embedding(config.vocab_size, config.hidden_size)
        self.layers = nn.ModuleList([Qwen3DecoderLayer(config)
                                     for _ in range(config.num_hidden_layers)])
        self.norm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)

    def forward(self, input_ids, positions, aux_layers=None):
        """aux_layers: layer indices whose incoming residual stream is also returned
        (concatenated, [N, len(aux_layers) * hidden]) -- the EAGLE-3 target features."""
        hidden_states = self.embed_tokens(input_ids)
        residual = None
        captured = {}
        for i, layer in enumerate(self.layers):
            aux = [] if aux_layers and i in aux_layers else None
            hidden_states, residual = layer(positions, hidden_states, residual, aux)
            if aux:
                captured[i] = aux[0]
        hidden_states, _ = self.norm(hidden_states, residual)
        if not aux_layers:
            return hidden_states
        return hidden_states, torch.cat([captured[i] for i in aux_layers], dim=-1)


class Qwen3ForCausalLM(nn.Module):

    def __init__(self, config):
        super().__init__()
        self.model = Qwen3Model(config)
        self.lm_head = nn.Linear(config.hidden_size, config.vocab_size, bias=False)
        if getattr(config, "tie_word_embeddings", False):
            self.lm_head.weight = self.model.embed_tokens.weight

    def forward(self, input_ids, positions, aux_layers=None):
        return self.model(input_ids, positions, aux_layers)

    def compute_logits(self, hidden_states):
        return self.lm_head(hidden_states)

    def attention_layers(self):
        return [m for m in self.modules() if isinstance(m, Attention)]


def random_init_(model, std=0.02, seed=0):
    """Random-init every weight in place (N(0, std); norms at 1)."""
    gen = torch.Generator(device=next(model.parameters()).device).manual_seed(seed)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("norm.weight"):
                p.fill_(1.0)
            else:
                p.normal_(0.0, std, generator=gen)
    return model


def qwen3_config(name):
    """Public Qwen3 architecture shapes (no checkpoint needed)."""
    from transformers import Qwen3Config
    shapes = {
        "Qwen3-8B": dict(hidden_size=4096, intermediate_size=12288, num_hidden_layers=36,
                         num_attention_heads=32, num_key_value_heads=8, head_dim=128,
                         vocab_size=151936, max_position_embeddings=40960, rope_theta=1000000,
                         rms_norm_eps=1e-6, tie_word_embeddings=False),
        "Qwen3-0.6B": dict(hidden_size=1024, intermediate_size=3072, num_hidden_layers=28,
                           num_attention_heads=16, num_key_value_heads=8, head_dim=128,
                           vocab_size=151936, max_position_embeddings=40960, rope_theta=1000000,
                           rms_norm_eps=1e-6, tie_word_embeddings=True),
    }
    cfg = Qwen3Config(**shapes[name], hidden_act="silu", attention_bias=False)
    cfg.dtype = torch.bfloat16
    return cfg
