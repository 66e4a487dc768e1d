"""Fused model layers (HIP) vs plain PyTorch fp32 restatements of the reference
layers (layernorm.py:16-40, rotary_embedding.py:6-14, activation.py:8-11) and of
the KV store (attention.py:21-30)."""
import pytest
import torch

from nanovllm.layers.activation import silu_and_mul
from nanovllm.layers.layernorm import rms_norm
from nanovllm.layers.rotary_embedding import RotaryEmbedding
from nanovllm import _C


def ref_rms(x, w, eps, residual=None):
    x = x.float()
    if residual is not None:
        x = x + residual.float()
        residual = x.to(torch.bfloat16)
    var = x.pow(2).mean(-1, keepdim=True)
    y = (x * torch.rsqrt(var + eps)).to(torch.bfloat16)
    y = (y.float() * w.float()).to(torch.bfloat16)
    return y if residual is None else (y, residual)


def ulps(a, b):
    """Distance in bf16 ulps (both bf16)."""
    ai = a.view(torch.int16).int()
    bi = b.view(torch.int16).int()
    ai = torch.where(ai < 0, -(ai & 0x7fff), ai)
    bi = torch.where(bi < 0, -(bi & 0x7fff), bi)
    return (ai - bi).abs()


@pytest.mark.gpu
# Hidden sizes of the Qwen3 family and two others, 257 rows each.
@pytest.mark.parametrize("H", [4096, 3072, 2048, 1024, 1536, 128])
def test_rmsnorm_plain_and_add(dev, H):
    g = torch.Generator().manual_seed(H)
    x = torch.randn(257, H, generator=g).to(torch.bfloat16)
    r = torch.randn(257, H, generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16)
    # the normalised value is rounded to bf16 before the weight multiply (as in the
    # reference), so a 1-ulp difference in rsqrt can surface as 2 ulps
    y = rms_norm(x.to(dev), w.to(dev), 1e-6).cpu()
    d = ulps(y, ref_rms(x, w, 1e-6))
    assert d.max() <= 2 and d.float().mean() < 0.05
    y2, r2 = rms_norm(x.to(dev), w.to(dev), 1e-6, r.to(dev))
    ey, er = ref_rms(x, w, 1e-6, r)
    assert torch.equal(r2.cpu(), er)
    d = ulps(y2.cpu(), ey)
    assert d.max() <= 2 and d.float().mean() < 0.05


@pytest.mark.gpu
# Every thread count and pieces per thread of the launch: the last size of each, the next
# one up, the smallest and the largest; odd row counts, with a padded row stride.
@pytest.mark.parametrize("H,N", [(H, N) for H in (8, 1024, 1032, 2048, 2056, 4096, 4104, 5120, 8184, 8192)
                                 for N in (1, 5)] + [(3072, 8193), (3080, 8193)])
def test_rmsnorm_launch_edges(dev, H, N):
    g = torch.Generator().manual_seed(H + N)
    x = torch.randn(N, H + 8, generator=g).to(torch.bfloat16)
    r = torch.randn(N, H, generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16)
    xd = x.to(dev)[:, :H]
    y = rms_norm(xd, w.to(dev), 1e-6).cpu()
    y2, r2 = rms_norm(xd, w.to(dev), 1e-6, r.to(dev))
    ey, er = ref_rms(x[:, :H], w, 1e-6, r)
    assert torch.equal(r2.cpu(), er)
    # as above: a 1-ulp difference in rsqrt can surface as 2 ulps, rarely
    for got, want in ((y, ref_rms(x[:, :H], w, 1e-6)), (y2.cpu(), ey)):
        d = ulps(got, want)
        assert d.max() <= 2 and (d > 0).float().mean() < max(0.05, 2 / d.numel())


def ref_rope(x, pos, base=1000000.0):
    """NeoX rotate-half RoPE in fp32 (reference rotary_embedding.py:6-14), with the
    angles computed in float64 from the definition a = p * base^(-2j/D)."""
    D = x.shape[-1]
    j = torch.arange(D // 2, dtype=torch.float64)
    ang = pos.double()[:, None] * base ** (-2.0 * j / D)[None, :]
    cos, sin = ang.cos().float()[:, None, :], ang.sin().float()[:, None, :]
    x1, x2 = x.float().chunk(2, dim=-1)
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1).to(torch.bfloat16)


def run_qk_norm_rope(dev, qkv, qw, kw, pos, Hq, Hkv, rope, k_cache=None, v_cache=None,
                     slots=None, want_k=True):
    N, D = qkv.shape[0], 128
    # device copies are bound to names: a temporary freed after its pointer is taken
    # could be handed to the next allocation before the kernel runs
    qd = qkv.to(dev)
    kd = torch.empty(N, Hkv, D, dtype=torch.bfloat16, device=dev) if want_k else None
    q = torch.empty(N, Hq, D, dtype=torch.bfloat16, device=dev)
    cs, posd = rope.cos_sin_cache.to(dev), pos.to(dev)
    qwd = None if qw is None else qw.to(dev)
    kwd = None if kw is None else kw.to(dev)
    sd = None if slots is None else slots.to(dev)
    _C.check(_C.lib().nvx_qk_norm_rope(_C.ptr(qd), qd.stride(0), Hq, Hkv, D, _C.ptr(qwd),
                                       _C.ptr(kwd), _C.ptr(posd), _C.ptr(cs), rope.max_positions,
                                       N, _C.ptr(q), _C.ptr(kd), _C.ptr(k_cache), _C.ptr(v_cache),
                                       _C.ptr(sd), 1e-6, _C.stream_of(qd)))
    torch.cuda.synchronize()
    return q.cpu(), None if kd is None else kd.cpu()


def assert_rope_close(a, b):
    # RoPE mixes two rounded values (x1*cos - x2*sin), so outputs near zero can
    # differ by many ulps while the absolute error stays at bf16 resolution
    err = (a.float() - b.float()).abs()
    assert float(err.max()) < 3e-2, float(err.max())
    assert float((err / (b.float().abs() + 1e-2)).mean()) < 2e-3


@pytest.mark.gpu
# Head layouts of Qwen3-8B (32/8) and Qwen3-0.6B (16/8) and two others, with token
# counts that leave a partial last workgroup.
@pytest.mark.parametrize("N,Hq,Hkv", [(300, 8, 2), (301, 32, 8), (77, 16, 8), (50, 12, 4)])
def test_qk_norm_rope(dev, N, Hq, Hkv):
    g = torch.Generator().manual_seed(N)
    D = 128
    qkv = torch.randn(N, (Hq + 2 * Hkv) * D, generator=g).to(torch.bfloat16)
    qw = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16)
    kw = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16)
    pos = torch.randint(0, 5000, (N,), generator=g)
    rope = RotaryEmbedding(D, D, 8192, 1000000.0)
    q_ref = ref_rope(ref_rms(qkv[:, :Hq * D].reshape(N, Hq, D), qw, 1e-6), pos)
    k_ref = ref_rope(ref_rms(qkv[:, Hq * D:(Hq + Hkv) * D].reshape(N, Hkv, D), kw, 1e-6), pos)
    print(f"[qk_norm_rope] N={N} Hq={Hq} Hkv={Hkv}", flush=True)
    q, k = run_qk_norm_rope(dev, qkv, qw, kw, pos, Hq, Hkv, rope)
    assert_rope_close(q, q_ref)
    assert_rope_close(k, k_ref)


@pytest.mark.gpu
def test_qk_norm_rope_stores_kv_and_rope_only():
    """The fused store: k (rotated) and the raw v land at their slot rows, slot -1
    rows stay untouched, and k_out may be omitted.  Without norm weights only RoPE is
    applied (Llama-style heads)."""
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(5)
    N, Hq, Hkv, D, nblk, bs = 70, 16, 8, 128, 3, 256
    qkv = torch.randn(N, (Hq + 2 * Hkv) * D, generator=g).to(torch.bfloat16)
    pos = torch.randint(0, 3000, (N,), generator=g)
    perm = torch.randperm(nblk * bs, generator=g)[:N].to(torch.int32)
    slots = perm.clone()
    slots[::7] = -1
    rope = RotaryEmbedding(D, D, 4096, 1000000.0)
    init = torch.randn(nblk, bs, Hkv, D, generator=g).to(torch.bfloat16)
    kc, vc = init.clone().to(dev), init.clone().to(dev)
    print("[qk_norm_rope] store + rope only", flush=True)
    q, k = run_qk_norm_rope(dev, qkv, None, None, pos, Hq, Hkv, rope, kc, vc, slots, want_k=False)
    assert k is None
    q_ref = ref_rope(qkv[:, :Hq * D].reshape(N, Hq, D), pos)
    k_ref = ref_rope(qkv[:, Hq * D:(Hq + Hkv) * D].reshape(N, Hkv, D), pos)
    v_raw = qkv[:, (Hq + Hkv) * D:].reshape(N, Hkv, D)
    assert_rope_close(q, q_ref)
    kexp, vexp = init.clone().view(-1, Hkv, D), init.clone().view(-1, Hkv, D)
    live = slots >= 0
    kc_h, vc_h = kc.cpu().view(-1, Hkv, D), vc.cpu().view(-1, Hkv, D)
    assert torch.equal(vc_h[slots[live].long()], v_raw[live])
    assert_rope_close(kc_h[slots[live].long()], k_ref[live])
    untouched = torch.ones(nblk * bs, dtype=torch.bool)
    untouched[slots[live].long()] = False
    assert torch.equal(kc_h[untouched], kexp[untouched])
    assert torch.equal(vc_h[untouched], vexp[untouched])
    # with norm weights and k_out as well: the cache rows equal k_out bit for bit
    qw = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16)
    kw = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16)
    _, k2 = run_qk_norm_rope(dev, qkv, qw, kw, pos, Hq, Hkv, rope, kc, vc, slots)
    assert torch.equal(kc.cpu().view(-1, Hkv, D)[slots[live].long()], k2[live])


@pytest.mark.gpu
def test_qk_norm_rope_position_outside_table_is_nan():
    """Positions past the RoPE table poison their token's outputs (NaN) instead of
    reading out of bounds; other tokens are unaffected."""
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(6)
    N, Hq, Hkv, D = 8, 4, 2, 128
    qkv = torch.randn(N, (Hq + 2 * Hkv) * D, generator=g).to(torch.bfloat16)
    rope = RotaryEmbedding(D, D, 512, 1000000.0)
    pos = torch.tensor([0, 511, 512, -1, 5, 1 << 40, 100, 511])
    print("[qk_norm_rope] positions outside the table", flush=True)
    q, k = run_qk_norm_rope(dev, qkv, None, None, pos, Hq, Hkv, rope)
    bad = torch.tensor([False, False, True, True, False, True, False, False])
    assert torch.isnan(q[bad].float()).all() and torch.isnan(k[bad].float()).all()
    assert not torch.isnan(q[~bad].float()).any() and not torch.isnan(k[~bad].float()).any()
    assert_rope_close(q[~bad], ref_rope(qkv[:, :Hq * D].reshape(N, Hq, D), pos.clamp(0, 511))[~bad])


@pytest.mark.gpu
def test_silu_mul(dev):
    g = torch.Generator().manual_seed(1)
    x = (torch.randn(129, 2 * 3072, generator=g) * 3).to(torch.bfloat16)
    out = silu_and_mul(x.to(dev)).cpu()
    gte, up = x.float().chunk(2, -1)
    ref = (torch.nn.functional.silu(gte) * up).to(torch.bfloat16)
    d = ulps(out, ref)
    assert d.max() <= 1 and d.float().mean() < 0.05
