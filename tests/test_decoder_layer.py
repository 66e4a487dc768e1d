"""The decoder layer's step over few rows (nvx_skinny_gemm, nvx_decoder_layer) against
plain fp32 products and the layer's modules run one by one."""
import ctypes

import numpy as np
import pytest
import torch

from nanovllm import _C
from nanovllm.layers.decoder import few_rows_layer
from nanovllm.models.qwen3 import Qwen3Attention, Qwen3DecoderLayer, Qwen3MLP, random_init_
from nanovllm.spec.tree import ancestor_masks, random_tree
from nanovllm.utils.context import get_context, reset_context, set_context
from nanovllm.utils.synthetic import paged_block_tables, slots_for


def test_validation_errors_are_reported():
    L = _C.lib()
    h = ctypes.c_void_p(0x100000)  # non-null host addresses: refused before any launch
    assert L.nvx_skinny_gemm(h, 64, h, h, 33, 16, 64, 0, None) == -1
    assert b"rows" in L.nvx_last_error()
    assert L.nvx_skinny_gemm(h, 96, h, h, 1, 16, 96, 0, None) == -1
    assert b"multiple" in L.nvx_last_error()
    assert L.nvx_skinny_gemm(h, 32, h, h, 1, 16, 64, 0, None) == -1
    assert b"row stride" in L.nvx_last_error()
    a = _C.DecoderLayerArgs(num_tokens=1, hidden_size=64, inter_size=64, num_heads=2, num_kv_heads=1,
                            head_dim=128, num_seqs=1, max_seqlen_q=1, max_context_len=64)
    need = L.nvx_decoder_layer_scratch_size(ctypes.byref(a))
    assert need > 0
    assert L.nvx_decoder_layer(ctypes.byref(a), h, need - 1, None) == -1
    assert b"scratch" in L.nvx_last_error()


@pytest.mark.gpu
# Rows at the edges of the groups of 8; columns and contraction lengths on both sides of
# every tile width, fewer blocks than waves and uneven shares among them.
@pytest.mark.parametrize("rows", [1, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(8, 64), (24, 320), (3072, 192), (3080, 64), (4096, 576), (6144, 128),
                                 (6160, 64), (2288, 128), (2304, 64), (4576, 64), (4608, 128)])
@pytest.mark.parametrize("silu", [0, 1])
def test_skinny_gemm(dev, rows, n, k, silu):
    g = torch.Generator().manual_seed(rows * 7 + n + k)
    pad = torch.randn(rows, k + 64, generator=g).to(torch.bfloat16).to(dev)  # row stride k + 64
    x = pad[:, :k]
    w = (torch.randn(n * (1 + silu), k, generator=g) * k ** -0.5).to(torch.bfloat16).to(dev)
    out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    _C.check(_C.lib().nvx_skinny_gemm(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), rows, n,
                                      k, silu, _C.stream_of(x)))
    y = x.double() @ w.double().T
    scale = x.double().abs() @ w.double().abs().T  # bounds the fp32 sums' error
    if silu:
        gate, up = y.split(n, 1)
        y = torch.nn.functional.silu(gate) * up
        sg, su = scale.split(n, 1)
        scale = (1.1 * sg) * up.abs() + gate.abs() * su  # |silu'| <= 1.1
    err = (out[:rows].double() - y).abs()
    # one rounding to bf16, k fp32 additions, expf and the division to a few ulps
    assert (err <= y.abs() * 2.0 ** -8 + scale * (k + 16) * 2.0 ** -23).all()
    assert (out[rows] == 7.0).all()  # nothing past the last row


def _step(layer, hidden, residual, nodes, ctx, dev, seed):
    """A step's context, positions and caches: `nodes` rows for each context length."""
    rng = np.random.default_rng(seed)
    B = len(ctx)
    bt, nblk = paged_block_tables(np.array(ctx) + nodes, 256, rng)
    g = torch.Generator().manual_seed(seed)
    cache = torch.randn(2, nblk, 256, 2, 128, generator=g).to(torch.bfloat16).to(dev)
    layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = cache[0], cache[1]
    masks = None
    if nodes > 1:
        masks = np.concatenate([ancestor_masks(random_tree(nodes, min(3, nodes - 1), rng)) for _ in ctx])
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a, dtype=d)).to(dev)  # noqa: E731
    set_context(False, cu_seqlens_q=t(np.arange(B + 1) * nodes, np.int32), max_seqlen_q=nodes,
                slot_mapping=t(np.concatenate([slots_for(bt[b], ctx[b] + np.arange(nodes), 256)
                                               for b in range(B)]), np.int32),
                context_lens=t(np.array(ctx) + nodes, np.int32), block_tables=t(bt, np.int32),
                max_context_len=max(ctx) + nodes, tree_mask=None if masks is None else t(masks, np.int64))
    return t(np.concatenate([c + np.arange(nodes) for c in ctx]), np.int64), cache


def _layer(dev, hidden=512, inter=1536, qk_norm=True):
    from transformers import Qwen3Config
    cfg = Qwen3Config(hidden_size=hidden, intermediate_size=inter, num_hidden_layers=1,
                      num_attention_heads=4, num_key_value_heads=2, head_dim=128, vocab_size=512,
                      max_position_embeddings=4096, rope_theta=1000000, rms_norm_eps=1e-6,
                      hidden_act="silu", attention_bias=False)
    torch.set_default_dtype(torch.bfloat16)  # the rotary table stays fp32
    try:
        layer = Qwen3DecoderLayer(cfg)
        if not qk_norm:
            layer.self_attn = Qwen3Attention(hidden, 4, 2, max_position=4096, head_dim=128,
                                             rope_theta=1000000, qk_norm=False)
    finally:
        torch.set_default_dtype(torch.float32)
    return random_init_(layer.to(dev), std=0.05)


@pytest.mark.gpu
@pytest.mark.parametrize("ctx,nodes", [([300], 1), ([5, 700, 90], 1), ([40, 0, 513, 64], 5),
                                       ([130] * 32, 1)])
@pytest.mark.parametrize("first", [False, True])
def test_layer_matches_its_modules(dev, ctx, nodes, first):
    layer, N = _layer(dev), len(ctx) * nodes
    g = torch.Generator().manual_seed(N)
    hidden = torch.randn(N, 512, generator=g).to(torch.bfloat16).to(dev)
    residual = None if first else torch.randn(N, 512, generator=g).to(torch.bfloat16).to(dev)
    got, aux = [], [[], []]
    try:
        for i in (0, 1):
            positions, cache = _step(layer, hidden, residual, nodes, ctx, dev, 3)
            with torch.set_grad_enabled(i == 1):  # gradients: module by module
                used = few_rows_layer(layer, Qwen3Attention, Qwen3MLP, positions, hidden, residual)
                assert (used is None) == (i == 1)
                got.append((*layer(positions, hidden, residual, aux[i]), cache))
    finally:
        reset_context()
    assert torch.equal(aux[0][0], aux[1][0])
    # a dozen roundings to bf16 (2^-9 each) meet in the outputs, the projections' sums being
    # the only difference: a few per mille
    for a, b in zip(*got):
        a, b = a.detach().double(), b.detach().double()
        assert ((a - b).norm() / b.norm()) < 1e-2


@pytest.mark.gpu
def test_modules_run_where_something_watches_or_replaces_them(dev):
    layer = _layer(dev)
    hidden = torch.randn(2, 512).to(torch.bfloat16).to(dev)
    try:
        with torch.no_grad():
            positions, _ = _step(layer, hidden, None, 1, [30, 50], dev, 1)
            call = lambda h=hidden: few_rows_layer(layer, Qwen3Attention, Qwen3MLP, positions, h, None)  # noqa: E731
            assert call() is not None
            seen = []
            hook = layer.mlp.down_proj.register_forward_hook(lambda *a: seen.append(1))
            assert call() is None
            layer(positions, hidden, None)
            assert seen
            hook.remove()
            assert call() is not None
            assert call(hidden.float()) is None
            assert call(torch.randn(33, 512, device=dev).to(torch.bfloat16)) is None
            layer.self_attn.o_proj = torch.nn.Sequential(layer.self_attn.o_proj)
            assert call() is None
    finally:
        reset_context()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["self_attn", "mlp"])
def test_replaced_blocks_run_as_modules(dev, name):
    """A wrapped attention or MLP block has none of the plain one's submodules."""
    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *args):
            return self.inner(*args)

    layer = _layer(dev)
    hidden = torch.randn(2, 512).to(torch.bfloat16).to(dev)
    try:
        positions, _ = _step(layer, hidden, None, 1, [30, 50], dev, 1)
        with torch.no_grad():
            wrapped = Wrapped(getattr(layer, name))
            setattr(layer, name, wrapped)
            assert few_rows_layer(layer, Qwen3Attention, Qwen3MLP, positions, hidden, None) is None
            out, residual = layer(positions, hidden, None)
            setattr(layer, name, wrapped.inner)
        with torch.enable_grad():  # the plain layer, module by module
            want, want_residual = layer(positions, hidden, None)
        assert torch.equal(out, want) and torch.equal(residual, want_residual)
    finally:
        reset_context()


@pytest.mark.gpu
# As serving runs every layer after the first: the residual stream between the norms stays
# in the call's scratch (no aux list).  Decode, tree and prefill contexts (there max_seqlen_k
# gives the longest context and a mask is dropped), layers with and without q/k norm.
@pytest.mark.parametrize("ctx,nodes,prefill,qk_norm", [
    ([5, 700, 90], 1, False, True), ([40, 0, 513, 64], 5, False, True), ([40, 0, 513], 5, False, False),
    ([0, 300], 16, True, True), ([7], 9, True, False)])
def test_layer_without_aux(dev, ctx, nodes, prefill, qk_norm):
    layer, N = _layer(dev, qk_norm=qk_norm), len(ctx) * nodes
    g = torch.Generator().manual_seed(N)
    hidden, residual = (torch.randn(N, 512, generator=g).to(torch.bfloat16).to(dev) for _ in range(2))
    got = []
    try:
        for grad in (False, True):  # gradients: module by module
            positions, cache = _step(layer, hidden, residual, nodes, ctx, dev, 3)
            c = get_context()
            if prefill:
                set_context(True, cu_seqlens_q=c.cu_seqlens_q, max_seqlen_q=nodes,
                            max_seqlen_k=c.max_context_len, slot_mapping=c.slot_mapping,
                            context_lens=c.context_lens, block_tables=c.block_tables,
                            tree_mask=c.tree_mask)
            before, slots = cache.clone(), get_context().slot_mapping.long()
            with torch.set_grad_enabled(grad):
                assert (few_rows_layer(layer, Qwen3Attention, Qwen3MLP, positions, hidden, residual)
                        is None) == grad
                out, res = layer(positions, hidden, residual)
            got.append((out.detach(), res.detach(), cache.view(2, -1, 256)[:, slots]))
            kept = torch.ones(cache[0].numel() // 256, dtype=torch.bool, device=dev)
            kept[slots] = False
            assert torch.equal(cache.view(2, -1, 256)[:, kept], before.view(2, -1, 256)[:, kept])
    finally:
        reset_context()
    for a, b in zip(got[0][:2], got[1][:2]):  # a dozen roundings to bf16, as above
        assert ((a.double() - b.double()).norm() / b.double().norm()) < 1e-2
    # each new K and V row (both heads): a projection, the norm and the rotation, three
    # roundings to bf16 after sums in another order
    a, b = got[0][2].double(), got[1][2].double()
    assert ((a - b).norm(dim=2) <= 1e-2 * b.norm(dim=2)).all()


@pytest.mark.gpu
def test_rows_the_call_leaves_to_the_modules(dev):
    """17 to 32 rows above hidden 2,048, and a call under autocast."""
    try:
        with torch.no_grad():
            for hidden, rows, used in ((2048, 32, True), (2112, 16, True), (2112, 17, False)):
                layer = _layer(dev, hidden, 256)
                x = torch.randn(rows, hidden, device=dev).to(torch.bfloat16)
                positions, _ = _step(layer, x, None, 1, [30] * rows, dev, 1)
                call = lambda: few_rows_layer(layer, Qwen3Attention, Qwen3MLP, positions, x, None)  # noqa: E731
                assert (call() is not None) == used
                with torch.autocast("cuda", dtype=torch.bfloat16):
                    assert call() is None
    finally:
        reset_context()
