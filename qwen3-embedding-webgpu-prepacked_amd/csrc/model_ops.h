// model_ops.h -- launchers of the row-wise model kernels (model_ops.hip) and their limits.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attn_common.h"
#include "qk_rope.h"

namespace qattn {

constexpr int kQ6KBlockBytes = 210;   // GGML Q6_K: 256 values (ggml block_q6_K)
constexpr int kRmsMaxWidth = 4096;    // rmsnorm_kernel: columns per row (one wavefront, 8 per lane per pass)

// out[t][c] (c < width, a multiple of 256) = token ids[t]'s row of the Q6_K table of `vocab` rows;
// ids outside [0, vocab) give zero rows.
hipError_t launch_embed_q6k(const int32_t* ids, int64_t tokens, const uint8_t* table, int64_t vocab, int width,
                            half_t* out, int64_t out_stride, hipStream_t stream);
// Residual add (residual may be NULL) + RMSNorm of `rows` rows of `width` (multiple of 8, <= kRmsMaxWidth).
hipError_t launch_rmsnorm(half_t* x, const half_t* residual, const float* weight, half_t* out, int64_t rows,
                          int width, int64_t x_stride, int64_t r_stride, int64_t out_stride, float eps,
                          hipStream_t stream);
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
// Residual add + RMSNorm of one row (RmsNormKernel, ops.ts:21-72), one wavefront; lane l owns columns
// 8l + 512j.  With a residual row rr: v = f32(x) + f32(r), x_out <- f16(v) (ops.ts:41; x_out may be xr,
// or NULL to leave it), and the sum of squares takes the unrounded v (ops.ts:42); without: v = f32(x).
// put(c, v) receives the normalised columns c..c+7: f16(f32(x) * inv * w) with the rounded x and
// inv = 1 / sqrt(sum / width + eps) (ops.ts:52-55).  The one formula of rmsnorm_kernel and of the
// projections that normalise their own rows, so the two agree bit for bit.
template <typename Put>
__device__ inline void rmsnorm_row(const half_t* xr, const half_t* rr, half_t* x_out, const float* weight, Put put,
                                   int width, float eps, int lane) {
  constexpr int kMaxChunks = kRmsMaxWidth / 512;
  half8 xs[kMaxChunks];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kMaxChunks; ++j) {
    const int c = 8 * lane + 512 * j;
    if (c < width) {
      half8 a = *reinterpret_cast<const half8*>(xr + c);
      if (rr) {
        const half8 b = *reinterpret_cast<const half8*>(rr + c);
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          s[e] = (float)a[e] + (float)b[e];
          a[e] = (half_t)s[e];
        }
        // The row's first pair adds its squares the other way round: the order (and so the rounding) of
        // embeddings stored before there was a fused projection.
        if (j == 0) ss = fmaf(s[0], s[0], s[1] * s[1]);
#pragma unroll
        for (int e = j == 0 ? 2 : 0; e < 8; ++e) ss = fmaf(s[e], s[e], ss);
        if (x_out) *reinterpret_cast<half8*>(x_out + c) = a;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf((float)a[e], (float)a[e], ss);
      }
      xs[j] = a;
    }
  }
  ss = wave_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)width + eps);
#pragma unroll
  for (int j = 0; j < kMaxChunks; ++j) {
    const int c = 8 * lane + 512 * j;
    if (c < width) {
      const float4 w0 = *reinterpret_cast<const float4*>(weight + c);
      const float4 w1 = *reinterpret_cast<const float4*>(weight + c + 4);
      const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      half8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = (float)xs[j][e] * inv * w[e];
        asm volatile("" : "+v"(v));  // rounded to fp32, then to fp16, in every caller (as swiglu_value)
        o[e] = (half_t)v;
      }
      put(c, o);
    }
  }
}

// ---- the small forward's fused projections (q4_matmul.hip), up to kFusedTokens tokens.
constexpr int kFusedTokens = 32;
// The rows a projection normalises itself: out-of-place residual add + RMSNorm of x (T x 1024).
struct FusedNorm {
  const half_t* x;
  const half_t* residual;  // NULL: no residual, x_out unused
  half_t* x_out;           // x + residual (another buffer than x: other workgroups still read it)
  const float* weight;
  float eps;
  int32_t tokens;
};
constexpr int kFusedSeqs = 64;
// Where the QKV projection's heads go, as qattn_qk_norm_rope_qkv leaves them: roped Q and K, V in
// its qkvRaw columns.
struct FusedQkv {
  half_t *q, *k, *qkv;  // row strides 2048, 1024, 4096
  const float *weight_q, *weight_k;
  const float2* rope;
  float eps;
  int32_t nseq;
  int32_t cu[kFusedSeqs + 1];
};
// RMSNorm + QKV projection + QK norm + RoPE (weight 1024 -> 4096) and RMSNorm + gate/up projection
// + SwiGLU (1024 -> 2 n_inter): bit for bit the separate launches.
hipError_t launch_q4_norm_qkv(const FusedNorm& n, const uint8_t* w, uint32_t w_bytes, const FusedQkv& out,
                              hipStream_t stream);
hipError_t launch_q4_norm_swiglu(const FusedNorm& n, const uint8_t* w, uint32_t w_bytes, int n_inter, half_t* y,
                                 int64_t ldy, hipStream_t stream);

// silu(g) * u in fp32, rounded to fp16: the one formula of swiglu_kernel and of the fused
// gate/up projection (q4_matmul.hip), so the two paths agree bit for bit.  The hardware exp2 and
// reciprocal (about 1 fp32 ulp each) are far inside the fp16 rounding of the result.
__device__ inline half_t swiglu_value(half_t g, half_t u) {
  const float gf = (float)g;
  float v = gf * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gf * -1.44269504f)) * (float)u;
  // The product is rounded to fp32 and then to fp16 in every caller: without this the compiler
  // may fold the multiply and the conversion into one v_fma_mix (a single rounding) in one
  // kernel and not in another.
  asm volatile("" : "+v"(v));
  return (half_t)v;
}

// out = silu(gate) * up for rows of [gate (width) | up (width)], width a multiple of 8.
hipError_t launch_swiglu(const half_t* gate_up, int64_t gu_stride, half_t* out, int64_t out_stride, int64_t rows,
                         int width, hipStream_t stream);

}  // namespace qattn
