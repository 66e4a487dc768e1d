// A decoder layer's step over few rows (decode and short verify steps), as one call.
//
// With a handful of rows every projection streams its weights once and does next to no
// arithmetic per byte, so the layer is bound by HBM -- or, for small models, by the
// launches themselves.  skinny_gemm_kernel computes y = x . W^T for at most 32 rows of x
// and nvx_decoder_layer enqueues the layer's kernels back to back from one host call:
//   add+RMSNorm, qkv, q/k norm + RoPE + KV store, attention, o_proj, add+RMSNorm,
//   gate_up with SiLU-mul, down.
#include "nvx_internal.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxRows = 32;  // rows of x: four groups of 8
constexpr int kKB = 64;       // one wave's block of the contraction: 128 bytes of a row of W
constexpr int kWaves = 4;      // waves that share a workgroup's contraction

__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// A workgroup computes NP groups of 8 outputs for up to 8*MG rows of x; its waves take the
// blocks of kKB elements of the contraction in turn and add their partial sums through
// LDS at the end (in wave order).  kSilu: each group comes with the same 8 columns of up
// (rows n and N + n of W), and y = silu(gate) * up.
//
// Every load takes whole 128-byte lines: 8 rows of W (or x) times kKB elements, lane l
// the 16-byte piece l/16 + 4*((l/8)%2) of row l%8.  As operands of
// v_mfma_f32_16x16x32_bf16 such a register holds the block's first 32 elements in rows
// (or columns) 0..7 and its last 32 in 8..15, so one product of a W and an x register
// gives both halves' sums in the two diagonal 8x8 quarters, which are added at the end;
// the off-diagonal quarters are not used.  (Fragments of 16 rows fetch half lines: with
// them a CU took in 22 B/ns, x included, and a 4096 x 12288 projection of 16 rows 29 us.)
// W is read exactly once, so LDS staging would only add a hop; x comes from L2.  U blocks
// are in flight while the U before are multiplied.  The loads are buffer loads: blocks
// past the end of the contraction and rows past M get an offset outside the buffer,
// which reads as zero without touching memory, so the loop has no branches that would
// make the compiler wait for loads early.
template <int MG, int NP, bool kSilu, int U>
__global__ __launch_bounds__(kWaves * 64) void skinny_gemm_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ W,
    uint16_t* __restrict__ out, int M, int N, int K) {
  constexpr int NT = kSilu ? 2 * NP : NP;  // group t: columns n0 + 8 * (t % NP), up rows from t = NP
  constexpr int kOutside = 0x7fffff00, kRsrcWord3 = 0x00020000, kNonTemporal = 2;
  extern __shared__ f32x4 red[];  // [waves][NT][MG][64]
  constexpr int nw = kWaves;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 7, piece = ((lane >> 4) + ((lane & 8) >> 1)) * 16;
  const int n0 = blockIdx.x * (8 * NP);
  __amdgpu_buffer_rsrc_t wr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wr[t] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(W + (int64_t)(n0 + (t % NP) * 8 + (t / NP) * N) * K), 0, 8 * K * 2,
        kRsrcWord3);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(x), 0, (int)(((M - 1) * x_stride + K) * 2), kRsrcWord3);
  const int w_off = r * K * 2 + piece;
  int x_off[MG];
#pragma unroll
  for (int m = 0; m < MG; ++m)
    x_off[m] = m * 8 + r < M ? (int)((m * 8 + r) * x_stride * 2) + piece : kOutside;
  const int nblk = K / kKB;  // this wave's blocks: wave, wave + nw, ...

  f32x4 acc[NT][MG];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MG; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct Buf {
    uint4 w[U][NT], x[U][MG];
  };
  auto load = [&](int b, Buf& f) {  // blocks b, b + nw, ..
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int blk = b + u * nw;
      const int k = blk < nblk ? blk * (kKB * 2) : 0;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        f.w[u][t] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(wr[t], blk < nblk ? w_off : kOutside, k,
                                                         kNonTemporal));
#pragma unroll
      for (int m = 0; m < MG; ++m)
        f.x[u][m] = __builtin_bit_cast(
            uint4,
            __builtin_amdgcn_raw_buffer_load_b128(xr, blk < nblk ? x_off[m] : kOutside, k, 0));
    }
  };
  auto mul = [&](const Buf& f) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MG; ++m)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, f.w[u][t]), __builtin_bit_cast(bf16x8, f.x[u][m]), acc[t][m],
              0, 0, 0);
  };
  Buf f0, f1;
  load(wave, f0);
  for (int b = wave; b < nblk; b += 2 * U * nw) {
    load(b + U * nw, f1);
    __builtin_amdgcn_sched_barrier(0);  // loads go out before the products wait for theirs
    mul(f0);
    load(b + 2 * U * nw, f0);
    __builtin_amdgcn_sched_barrier(0);
    mul(f1);
  }

#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MG; ++m) red[((wave * NT + t) * MG + m) * 64 + lane] = acc[t][m];
  __syncthreads();
  // Lane l holds column l%16 (x row) and rows 4*(l/16) .. +3 (W rows) of the tile: the
  // first half's sums are in lanes of columns and rows 0..7, the second half's 40 lanes on.
  const int g = lane >> 4;
  if (g >= 2 || (lane & 8)) return;
  for (int i = wave; i < NP * MG; i += nw) {
    const int m = i % MG, p = i / MG;
    if (m * 8 + r >= M) continue;
    f32x4 s[kSilu ? 2 : 1];
#pragma unroll
    for (int h = 0; h < (kSilu ? 2 : 1); ++h) {
      const f32x4* t = red + ((p + h * NP) * MG + m) * 64 + lane;
      s[h] = t[0] + t[40];
      for (int w = 1; w < nw; ++w) s[h] += t[w * NT * MG * 64] + t[w * NT * MG * 64 + 40];
    }
    uint16_t y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v = s[0][j];
      if constexpr (kSilu) v = v / (1.f + __expf(-v)) * s[1][j];
      y[j] = f2bf(v);
    }
    *reinterpret_cast<uint2*>(out + (int64_t)(m * 8 + r) * N + n0 + p * 8 + 4 * g) =
        make_uint2((uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16));
  }
}

inline bool a16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <int MG, int NP, bool kSilu>
void launch_skinny(const void* x, int64_t x_stride, const void* w, void* out, int M, int N, int K,
                   hipStream_t s) {
  constexpr int U = MG * NP >= 8 ? 1 : 2;  // keeps two buffers within 128 registers
  const size_t lds = (size_t)kWaves * (kSilu ? 2 : 1) * NP * MG * 64 * sizeof(f32x4);
  hipLaunchKernelGGL((skinny_gemm_kernel<MG, NP, kSilu, U>), dim3(N / (8 * NP)), dim3(kWaves * 64), lds,
                     s, (const uint16_t*)x, x_stride, (const uint16_t*)w, (uint16_t*)out, M, N, K);
}

// Output columns per workgroup, 8 * NP.  A wider tile reads x fewer times, but a CU takes
// in only so many bytes at once, so the weights have to be spread over most of the 256 of
// them: the widest tile that leaves kBusy workgroups.  us per projection, [out, in]
// features, with 8, 16 and 32 columns per workgroup and hipBLASLt:
//   [2048, 6144],  8 rows:  8.3, 11.0, 16.3, 11.2;  16 rows: 11.0, 13.5, 19.5, 11.3
//   [2304, 9728],  8 rows: 20.4, 16.4, 24.6, 16.1;  16 rows: 28.9, 20.6, 28.8, 16.6
//   [4096, 9728],  8 rows: 21.4, 17.1, 25.3, 18.7;  16 rows: 29.8, 21.2, 29.8, 19.2
//   [4608, 4096], 16 rows: 19.5, 17.9, 14.6, 14.2
//   [6144, 4096], 16 rows: 20.2, 18.5, 15.7, 15.2;   8 rows: 15.0, 15.0, 15.6, 15.2
//   [4096, 12288], 16 rows: 35.8, 25.4, 37.9, 22.6;  8 rows: 28.9, 21.7, 34.7, 23.4
// One row is little x to read again: [3072, 9728] 15.2, 15.5; it keeps the narrow tile where
// the wider one does not reach every CU.  Up to 8 rows, 32 columns gain too little
// ([5632, 4096] 14.8, 14.4) to lose the smaller sums.  Gate/up, with 8 and 16 columns each:
//   [12288, 4096], 8 rows: 41.5, 37.2 (hipBLASLt, SiLU-mul not counted: 47.5)
//   [3072, 1024],  8 rows:  6.2,  5.8 (8.1)
constexpr int kBusy = 144, kCUs = 256;
template <int MG>
void launch_skinny_rows(const void* x, int64_t x_stride, const void* w, void* out, int M, int N, int K,
                        bool silu, hipStream_t s) {
  if (silu) {
    if (N % 16 == 0 && N / 16 >= 192)
      launch_skinny<MG, 2, true>(x, x_stride, w, out, M, N, K, s);
    else
      launch_skinny<MG, 1, true>(x, x_stride, w, out, M, N, K, s);
  } else {
    if (MG > 1 && N % 32 == 0 && N / 32 >= kBusy)
      launch_skinny<MG, 4, false>(x, x_stride, w, out, M, N, K, s);
    else if (N % 16 == 0 && N / 16 >= (M > 1 ? kBusy : kCUs))
      launch_skinny<MG, 2, false>(x, x_stride, w, out, M, N, K, s);
    else
      launch_skinny<MG, 1, false>(x, x_stride, w, out, M, N, K, s);
  }
}

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

struct Scratch {
  size_t normed, mid, qkv, q, o, proj, act, attn, total;
};

Scratch scratch_layout(const nvx_decoder_layer_args& a) {
  Scratch s;
  size_t at = 0;
  auto take = [&](size_t elems) {
    const size_t here = at;
    at += up256(elems * 2);
    return here;
  };
  const size_t n = (size_t)a.num_tokens;
  s.normed = take(n * a.hidden_size);
  s.mid = take(n * a.hidden_size);
  s.qkv = take(n * (a.num_heads + 2 * a.num_kv_heads) * a.head_dim);
  s.q = take(n * a.num_heads * a.head_dim);
  s.o = take(n * a.num_heads * a.head_dim);
  s.proj = take(n * a.hidden_size);
  s.act = take(n * a.inter_size);
  s.attn = at;
  s.total = at + nvx_tree_attention_workspace_size(a.num_seqs, a.num_tokens, a.max_seqlen_q,
                                                   a.max_context_len, a.num_heads, a.num_kv_heads,
                                                   a.head_dim);
  return s;
}

}  // namespace

extern "C" int nvx_skinny_gemm(const void* x, int64_t x_row_stride, const void* weight, void* out,
                               int32_t num_rows, int32_t out_features, int32_t in_features,
                               int32_t silu_mul, void* stream) {
  nvx::clear_error();
  NVX_CHECK(num_rows >= 0 && num_rows <= kMaxRows, "skinny_gemm: at most %d rows (got %d)", kMaxRows,
            num_rows);
  NVX_CHECK(out_features > 0 && out_features % 8 == 0 && in_features > 0 && in_features % kKB == 0,
            "skinny_gemm: out_features must be a multiple of 8 and in_features of %d (got %d, %d)",
            kKB, out_features, in_features);
  if (num_rows == 0) return NVX_OK;
  NVX_CHECK(x && weight && out && a16(x) && a16(weight) && a16(out) && x_row_stride % 8 == 0 &&
                x_row_stride >= in_features && x_row_stride < (1 << 24) && in_features < (1 << 24),
            "skinny_gemm: null or unaligned pointer, or a row stride out of range");
  hipStream_t s = (hipStream_t)stream;
  const bool silu = silu_mul != 0;
  if (num_rows <= 8)
    launch_skinny_rows<1>(x, x_row_stride, weight, out, num_rows, out_features, in_features, silu, s);
  else if (num_rows <= 16)
    launch_skinny_rows<2>(x, x_row_stride, weight, out, num_rows, out_features, in_features, silu, s);
  else
    launch_skinny_rows<4>(x, x_row_stride, weight, out, num_rows, out_features, in_features, silu, s);
  NVX_LAUNCHED();
  return NVX_OK;
}

extern "C" size_t nvx_decoder_layer_scratch_size(const nvx_decoder_layer_args* a) {
  return a && a->num_tokens > 0 ? scratch_layout(*a).total : 0;
}

extern "C" int nvx_decoder_layer(const nvx_decoder_layer_args* args, void* scratch,
                                 size_t scratch_bytes, void* stream) {
  nvx::clear_error();
  NVX_CHECK(args, "decoder_layer: null arguments");
  const nvx_decoder_layer_args& a = *args;
  NVX_CHECK(a.num_tokens >= 0 && a.num_tokens <= kMaxRows, "decoder_layer: at most %d rows (got %d)",
            kMaxRows, a.num_tokens);
  NVX_CHECK(a.hidden_size > 0 && a.hidden_size % kKB == 0 && a.inter_size > 0 &&
                a.inter_size % kKB == 0 && a.num_heads > 0 && a.num_kv_heads > 0 && a.head_dim == 128,
            "decoder_layer: hidden and intermediate sizes must be multiples of %d, head_dim 128", kKB);
  if (a.num_tokens == 0) return NVX_OK;
  const Scratch l = scratch_layout(a);
  NVX_CHECK(scratch && scratch_bytes >= l.total && ((uintptr_t)scratch & 255) == 0,
            "decoder_layer: 256-byte aligned scratch of %zu bytes required (got %zu)", l.total,
            scratch_bytes);
  char* const base = (char*)scratch;
  const int n = a.num_tokens, H = a.hidden_size, D = a.head_dim;
  const int qkv_cols = (a.num_heads + 2 * a.num_kv_heads) * D;
  // the residual stream entering the attention: hidden + residual, or hidden itself
  void* const mid = a.residual ? (a.residual_in_out ? a.residual_in_out : base + l.mid)
                               : const_cast<void*>(a.hidden);
#define NVX_STEP(call)            \
  do {                            \
    const int rc_ = (call);       \
    if (rc_ != NVX_OK) return rc_; \
  } while (0)
  NVX_STEP(nvx_rmsnorm(a.hidden, H, a.residual, a.residual ? mid : nullptr, a.input_norm,
                       base + l.normed, n, H, a.input_eps, stream));
  NVX_STEP(nvx_skinny_gemm(base + l.normed, H, a.qkv_weight, base + l.qkv, n, qkv_cols, H, 0, stream));
  NVX_STEP(nvx_qk_norm_rope(base + l.qkv, qkv_cols, a.num_heads, a.num_kv_heads, D, a.q_norm, a.k_norm,
                            a.positions, a.cos_sin_cache, a.cache_positions, n, base + l.q, nullptr,
                            a.k_cache, a.v_cache, a.slot_mapping, a.qk_eps, stream));
  NVX_STEP(nvx_tree_attention(base + l.q, base + l.o, a.k_cache, a.v_cache, a.block_tables,
                              a.block_table_stride, a.cu_seqlens_q, a.context_lens, a.tree_mask,
                              a.num_seqs, n, a.max_seqlen_q, a.max_context_len, a.num_heads,
                              a.num_kv_heads, D, a.block_size, a.scale, base + l.attn,
                              l.total - l.attn, stream));
  NVX_STEP(nvx_skinny_gemm(base + l.o, a.num_heads * D, a.o_weight, base + l.proj, n, H,
                           a.num_heads * D, 0, stream));
  NVX_STEP(nvx_rmsnorm(base + l.proj, H, mid, a.residual_out, a.post_norm, base + l.normed, n, H,
                       a.post_eps, stream));
  NVX_STEP(nvx_skinny_gemm(base + l.normed, H, a.gate_up_weight, base + l.act, n, a.inter_size, H, 1,
                           stream));
  NVX_STEP(nvx_skinny_gemm(base + l.act, a.inter_size, a.down_weight, a.out, n, H, a.inter_size, 0,
                           stream));
#undef NVX_STEP
  return NVX_OK;
}
