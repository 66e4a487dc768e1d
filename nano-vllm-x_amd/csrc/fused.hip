// Fused elementwise layers of the target model (bf16 in/out, fp32 math).
//
// These replace chains of eager torch kernels around the verify path's attention:
//   rmsnorm      : RMSNorm and add+RMSNorm   (reference nanovllm/layers/layernorm.py:16-40)
//   qk_norm_rope : per-head q/k RMSNorm then NeoX RoPE (qwen3.py:82-85,
//                  rotary_embedding.py:6-14, :37-48), writing contiguous q and
//                  storing k and v into the paged cache (attention.py:62-63)
//   silu_mul     : SiLU(gate) * up           (activation.py:8-11)
// Each is one pass over HBM: read the inputs once, write the outputs once.
#include "nvx_internal.h"

namespace {

__device__ __forceinline__ float bf(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float rbf(float x) { return bf(f2bf(x)); }  // round to bf16

// One workgroup per row; each thread owns 8-element (16-byte) pieces.
// plain: y = bf16(bf16(x * rsqrt(mean(x^2) + eps)) * w)
// add:   s = x + r (fp32); r_out = bf16(s); y from s as above.
// A decode step's few rows are bound by latency, not bytes: every load, the weight's too,
// is in flight before the sum of squares is reduced, and a row takes as many threads as it
// has pieces (kPer pieces each at most).  Add+RMSNorm, back to back: [8, 4096] 4.5 ->
// 3.5 us, [1, 1024] 3.1 -> 2.95 us, [16384, 1024] 25.8 -> 23.1 us against one 256-thread
// kernel that asked for the weight after the reduction.  That kernel is ahead at about
// 1,024 rows of 5,120 to 6,144 with a residual ([1024, 5120] 9.8, here 10.4), and behind at
// fewer and more rows ([256, 5120] 6.3, 5.1; [4096, 8192] 44.8, 42.1).
constexpr int kNormMaxHidden = 8192;
template <int NT, int kPer>
__global__ __launch_bounds__(NT) void rmsnorm_kernel(const uint16_t* __restrict__ x, int64_t x_stride,
                                                     const uint16_t* __restrict__ res,
                                                     uint16_t* __restrict__ res_out,
                                                     const uint16_t* __restrict__ w,
                                                     uint16_t* __restrict__ out, int H, float eps) {
  __shared__ float red[NT / nvx::kWave];
  const int row = blockIdx.x;
  const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)row * x_stride);
  const uint4* rr = res ? reinterpret_cast<const uint4*>(res + (int64_t)row * H) : nullptr;
  const uint4* wr = reinterpret_cast<const uint4*>(w);
  const int nv = H / 8;
  uint4 a[kPer], b[kPer], ww[kPer];
#pragma unroll
  for (int c = 0; c < kPer; ++c) {
    const int i = min((int)threadIdx.x + c * NT, nv - 1);
    a[c] = xr[i];
    b[c] = make_uint4(0, 0, 0, 0);
    if (rr) b[c] = rr[i];
    ww[c] = wr[i];
  }
  float v[kPer][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < kPer; ++c) {
    const int i = threadIdx.x + c * NT;
    if (i < nv) {
      const uint16_t* ah = reinterpret_cast<const uint16_t*>(&a[c]);
      const uint16_t* bh = reinterpret_cast<const uint16_t*>(&b[c]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float s = bf(ah[e]);
        if (rr) s = s + bf(bh[e]);
        v[c][e] = s;
        ss += s * s;
      }
      if (res_out) {
        uint4 o;
        uint16_t* oh = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
        for (int e = 0; e < 8; ++e) oh[e] = f2bf(v[c][e]);
        reinterpret_cast<uint4*>(res_out + (int64_t)row * H)[i] = o;
      }
    }
  }
  const float inv = rsqrtf(nvx::block_sum_any<NT>(ss, red) / (float)H + eps);
#pragma unroll
  for (int c = 0; c < kPer; ++c) {
    const int i = threadIdx.x + c * NT;
    if (i < nv) {
      const uint16_t* wh = reinterpret_cast<const uint16_t*>(&ww[c]);
      uint4 o;
      uint16_t* oh = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
      for (int e = 0; e < 8; ++e) oh[e] = f2bf(rbf(v[c][e] * inv) * bf(wh[e]));
      reinterpret_cast<uint4*>(out + (int64_t)row * H)[i] = o;
    }
  }
}

// Eight lanes per (token, head), 16-byte accesses: lane part p owns elements
// 8p..8p+7 and 64+8p..64+8p+7 -- the pairs NeoX RoPE rotates together (head_dim
// 128).  Heads 0..Hq-1 are q, Hq..Hq+Hkv-1 are k, and when the caches are given
// Hq+Hkv..Hq+2Hkv-1 are v, which is only copied to its cache row.
//   q, k: optional per-head RMSNorm (sum of squares reduced over the 8 lanes;
//         qw == nullptr skips it), then RoPE from the position's table row;
//   k, v: written to the cache row of slot_mapping[n] (skipped for slot -1), k
//         also to k_out when that is given.
// A position outside [0, max_pos) reads table row 0 and writes NaN, so a caller
// that runs past the table sees it in every output instead of reading out of
// bounds.
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(
    const uint16_t* __restrict__ qkv, int64_t row_stride, int Hq, int Hkv,
    const uint16_t* __restrict__ qw, const uint16_t* __restrict__ kw,
    const int64_t* __restrict__ positions, const float* __restrict__ cos_sin, int64_t max_pos,
    int N, uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out,
    uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping, float eps) {
  const int H = Hq + Hkv + (v_cache ? Hkv : 0);
  // (token, head); a 256-byte head each, so their number fits 32 bits
  const uint32_t unit = blockIdx.x * 32u + (threadIdx.x >> 3);
  const int part = threadIdx.x & 7;
  // Units are whole 8-lane groups, so a group is either fully in range or fully out.
  if (unit >= (uint32_t)N * (uint32_t)H) return;
  const int n = (int)(unit / (uint32_t)H), h = (int)(unit % (uint32_t)H);
  const uint16_t* src = qkv + (int64_t)n * row_stride + (int64_t)h * 128 + 8 * part;
  // Everything the unit needs is asked for at once; only the table row waits, for its
  // position (few rows are bound by these round trips: 8 rows of
  // 32/8 heads 3.8 us, 4.0 us with each load where it is used; 4,096 rows 23.8, 25.0 us).
  const int64_t pos = positions[n];
  const int32_t slot = k_cache && h >= Hq ? slot_mapping[n] : -1;
  const uint4 a = *reinterpret_cast<const uint4*>(src);
  const uint4 b = *reinterpret_cast<const uint4*>(src + 64);
  const bool isq = h < Hq;
  uint4 wa = make_uint4(0, 0, 0, 0), wb = wa;
  if (qw) {
    const uint16_t* w = (isq ? qw : kw) + 8 * part;
    wa = *reinterpret_cast<const uint4*>(w);
    wb = *reinterpret_cast<const uint4*>(w + 64);
  }
  const bool in_table = pos >= 0 && pos < max_pos;
  const float* cs = cos_sin + (in_table ? pos : 0) * 128 + 8 * part;
  const float4 c0 = *reinterpret_cast<const float4*>(cs);
  const float4 c1 = *reinterpret_cast<const float4*>(cs + 4);
  const float4 s0 = *reinterpret_cast<const float4*>(cs + 64);
  const float4 s1 = *reinterpret_cast<const float4*>(cs + 68);
  const int64_t kv_row = (int64_t)Hkv * 128;
  if (h >= Hq + Hkv) {  // v: a copy into the cache
    if (slot < 0) return;
    uint16_t* dst = v_cache + (int64_t)slot * kv_row + (int64_t)(h - Hq - Hkv) * 128 + 8 * part;
    *reinterpret_cast<uint4*>(dst) = a;
    *reinterpret_cast<uint4*>(dst + 64) = b;
    return;
  }
  const uint16_t* ah = reinterpret_cast<const uint16_t*>(&a);
  const uint16_t* bh = reinterpret_cast<const uint16_t*>(&b);
  float x1[8], x2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x1[e] = bf(ah[e]);
    x2[e] = bf(bh[e]);
  }
  if (qw) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += x1[e] * x1[e] + x2[e] * x2[e];
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) ss += nvx::shfl_xor_f(ss, off);
    const float inv = rsqrtf(ss / 128.f + eps);
    const uint16_t* wah = reinterpret_cast<const uint16_t*>(&wa);
    const uint16_t* wbh = reinterpret_cast<const uint16_t*>(&wb);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x1[e] = rbf(rbf(x1[e] * inv) * bf(wah[e]));
      x2[e] = rbf(rbf(x2[e] * inv) * bf(wbh[e]));
    }
  }
  const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
  uint4 oa, ob;
  uint16_t* oah = reinterpret_cast<uint16_t*>(&oa);
  uint16_t* obh = reinterpret_cast<uint16_t*>(&ob);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    oah[e] = f2bf(x1[e] * cv[e] - x2[e] * sv[e]);
    obh[e] = f2bf(x2[e] * cv[e] + x1[e] * sv[e]);
  }
  if (!in_table) {  // bf16 NaN poisons the row
    oa = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
    ob = oa;
  }
  if (isq) {
    uint16_t* dst = q_out + ((int64_t)n * Hq + h) * 128 + 8 * part;
    *reinterpret_cast<uint4*>(dst) = oa;
    *reinterpret_cast<uint4*>(dst + 64) = ob;
    return;
  }
  const int kh = h - Hq;
  if (k_out) {
    uint16_t* dst = k_out + ((int64_t)n * Hkv + kh) * 128 + 8 * part;
    *reinterpret_cast<uint4*>(dst) = oa;
    *reinterpret_cast<uint4*>(dst + 64) = ob;
  }
  if (slot >= 0) {
    uint16_t* dst = k_cache + (int64_t)slot * kv_row + (int64_t)kh * 128 + 8 * part;
    *reinterpret_cast<uint4*>(dst) = oa;
    *reinterpret_cast<uint4*>(dst + 64) = ob;
  }
}

// out[n, i] = bf16(silu(gate) * up), gate = gu[n, i], up = gu[n, I + i]; 8 per thread.
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu,
                                                       int64_t stride, uint16_t* __restrict__ out,
                                                       int N, int I) {
  const int nv = I / 8;
  const int64_t total = (int64_t)N * nv;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (int64_t)gridDim.x * 256) {
    const int n = (int)(t / nv), i = (int)(t - (int64_t)n * nv);
    const uint4 g = reinterpret_cast<const uint4*>(gu + (int64_t)n * stride)[i];
    const uint4 u = reinterpret_cast<const uint4*>(gu + (int64_t)n * stride + I)[i];
    const uint16_t* gh = reinterpret_cast<const uint16_t*>(&g);
    const uint16_t* uh = reinterpret_cast<const uint16_t*>(&u);
    uint4 o;
    uint16_t* oh = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = bf(gh[e]);
      oh[e] = f2bf(a / (1.f + __expf(-a)) * bf(uh[e]));
    }
    reinterpret_cast<uint4*>(out + (int64_t)n * I)[i] = o;
  }
}

inline bool a16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

extern "C" int nvx_rmsnorm(const void* x, int64_t x_row_stride, const void* residual,
                           void* residual_out, const void* weight, void* out, int32_t num_rows,
                           int32_t hidden, float eps, void* stream) {
  nvx::clear_error();
  NVX_CHECK(hidden > 0 && hidden % 8 == 0 && hidden <= kNormMaxHidden,
            "rmsnorm: hidden must be a multiple of 8 and <= %d (got %d)", kNormMaxHidden,
            hidden);
  NVX_CHECK(num_rows >= 0 && x_row_stride % 8 == 0, "rmsnorm: bad rows/stride");
  NVX_CHECK((residual == nullptr) == (residual_out == nullptr),
            "rmsnorm: residual and residual_out go together");
  if (num_rows == 0) return NVX_OK;
  NVX_CHECK(x && weight && out && a16(x) && a16(weight) && a16(out) &&
                (!residual || (a16(residual) && a16(residual_out))),
            "rmsnorm: null or unaligned pointer");
  hipStream_t s = (hipStream_t)stream;
#define NVX_NORM(NT, PER)                                                                       \
  hipLaunchKernelGGL((rmsnorm_kernel<NT, PER>), dim3(num_rows), dim3(NT), 0, s, (const uint16_t*)x, \
                     x_row_stride, (const uint16_t*)residual, (uint16_t*)residual_out,          \
                     (const uint16_t*)weight, (uint16_t*)out, hidden, eps)
  // 2,049 to 4,096: with a residual, a piece per thread (us with 256 threads of two and 512 of
  // one: [1024, 4096] 8.45, 7.95; [4096, 3072] 20.2, 18.8; [16384, 4096] 96.8, 92.3), unless
  // many rows leave a quarter of the threads idle ([16384, 2560] 61.6, 64.1); without a
  // residual, two pieces per thread stream many rows better ([16384, 4096] 41.2, 46.1).
  if (hidden <= 128 * 8)
    NVX_NORM(128, 1);
  else if (hidden <= 256 * 8)
    NVX_NORM(256, 1);
  else if (hidden <= 512 * 8 && residual && (hidden > 384 * 8 || num_rows <= 8192))
    NVX_NORM(512, 1);
  else if (hidden <= 512 * 8)
    NVX_NORM(256, 2);
  else
    NVX_NORM(512, 2);
#undef NVX_NORM
  NVX_LAUNCHED();
  return NVX_OK;
}

extern "C" int nvx_qk_norm_rope(const void* qkv, int64_t qkv_row_stride, int32_t num_q_heads,
                                int32_t num_kv_heads, int32_t head_dim, const void* q_norm_weight,
                                const void* k_norm_weight, const int64_t* positions,
                                const float* cos_sin_cache, int64_t cache_positions,
                                int32_t num_tokens, void* q_out, void* k_out, void* k_cache,
                                void* v_cache, const int32_t* slot_mapping, float eps,
                                void* stream) {
  nvx::clear_error();
  NVX_CHECK(head_dim == 128, "qk_norm_rope: head_dim must be 128 (got %d)", head_dim);
  NVX_CHECK(num_tokens >= 0 && num_q_heads > 0 && num_kv_heads > 0 && cache_positions > 0,
            "qk_norm_rope: bad sizes");
  NVX_CHECK((q_norm_weight == nullptr) == (k_norm_weight == nullptr),
            "qk_norm_rope: q_norm_weight and k_norm_weight go together (both NULL: no norm)");
  NVX_CHECK((k_cache == nullptr) == (v_cache == nullptr) &&
                (k_cache == nullptr) == (slot_mapping == nullptr),
            "qk_norm_rope: k_cache, v_cache and slot_mapping go together");
  NVX_CHECK(k_out || k_cache, "qk_norm_rope: k needs a destination (k_out or the caches)");
  if (num_tokens == 0) return NVX_OK;
  NVX_CHECK(qkv && positions && cos_sin_cache && q_out, "qk_norm_rope: null pointer");
  NVX_CHECK(a16(qkv) && (!q_norm_weight || (a16(q_norm_weight) && a16(k_norm_weight))) &&
                a16(cos_sin_cache) && a16(q_out) && (!k_out || a16(k_out)) &&
                (!k_cache || (a16(k_cache) && a16(v_cache))) && qkv_row_stride % 8 == 0,
            "qk_norm_rope: pointers must be 16-byte aligned and the row stride a multiple of 8");
  const int heads = num_q_heads + num_kv_heads + (v_cache ? num_kv_heads : 0);
  const int64_t lanes = (int64_t)num_tokens * heads * 8;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(qk_norm_rope_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, s,
                     (const uint16_t*)qkv, qkv_row_stride, num_q_heads, num_kv_heads,
                     (const uint16_t*)q_norm_weight, (const uint16_t*)k_norm_weight, positions,
                     cos_sin_cache, cache_positions, num_tokens, (uint16_t*)q_out,
                     (uint16_t*)k_out, (uint16_t*)k_cache, (uint16_t*)v_cache, slot_mapping, eps);
  NVX_LAUNCHED();
  return NVX_OK;
}

extern "C" int nvx_silu_mul(const void* gate_up, int64_t row_stride, void* out, int32_t num_rows,
                            int32_t inter, void* stream) {
  nvx::clear_error();
  NVX_CHECK(inter > 0 && inter % 8 == 0 && row_stride % 8 == 0 && num_rows >= 0,
            "silu_mul: inter and stride must be multiples of 8");
  if (num_rows == 0) return NVX_OK;
  NVX_CHECK(gate_up && out && a16(gate_up) && a16(out), "silu_mul: null or unaligned pointer");
  const int64_t work = (int64_t)num_rows * (inter / 8);
  int64_t grid = (work + 255) / 256;
  if (grid > 65536) grid = 65536;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)grid), dim3(256), 0, s,
                     (const uint16_t*)gate_up, row_stride, (uint16_t*)out, num_rows, inter);
  NVX_LAUNCHED();
  return NVX_OK;
}
