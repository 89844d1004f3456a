// qk_rope.h -- launch arguments of the QK-norm + RoPE producer (qk_rope.hip), shared with the
// host entry points that fill them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qattn {

typedef _Float16 half_t;

typedef half_t rope_h8 __attribute__((ext_vector_type(8)));
// The value of lane l ^ N (N = 8), or one equal to it where values already repeat every 2 N lanes, as in
// a sum over xor distances from 8 down: a rotation within the 16 lanes of a row, one VALU operation
// where a shuffle goes through LDS (us, shuffles -> this: QK norm + RoPE of 8,000 tokens, twelve of them
// per vector, 20.9 -> 20.1; forward of 15 tokens 1,024 -> 1,010, of 500 2,275 -> 2,241).
template <int N>
__device__ inline float row_rotate(float v) {
  const int i = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x120 + N, 0xf, 0xf, false));
}
// The sum over the 16 lanes of a row: xor distances 8, 4, 2, 1 in turn.
__device__ inline float row_sum(float v) {
  v += row_rotate<8>(v);
  v += row_rotate<4>(v);
  v += row_rotate<2>(v);
  return v + row_rotate<1>(v);
}
// The sum over the wavefront: xor distances 32, 16, then the row's.
__device__ inline float wave_sum(float v) {
  const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
  const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return row_sum(__uint_as_float(rows[0]) + __uint_as_float(rows[1]));
}

// QK RMSNorm + RoPE of one 128-wide head vector held by 16 lanes (lane j: elements 8j..8j+7) with gains
// g0, g1 and c4 = (cos, sin) of slots 8 (j & 7) .. +7 (ops.ts:125-147, f32).  The sum of squares is
// reduced over the 16 lanes in a fixed order; the rotate-half partner of element d
// (d +- 64) sits in lane j ^ 8 at the same slot.  The one formula of qk_norm_rope_kernel and of the
// fused small projection, so the two agree bit for bit.
// quad: the vector's place among a token's head vectors, in fours.
// A rotated element is fma(n, cos, partner * sin) rounded once to fp16, except elements 1-6 of the first
// four vectors and 2-7 of the second four: they round to fp32 and then to fp16, and every other one
// of them is fma(partner, sin, n * cos).  That is how the compiler once laid out the separate launch;
// it is spelled out so that embeddings stored before there was a fused projection stay equal bit for
// bit and no longer depend on the compiler.
template <int QUAD>
__device__ inline rope_h8 rope_rotate(const float (&n)[8], const float (&partner)[8], const float4 (&c4)[4]) {
  rope_h8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float4 c = c4[e >> 1];  // (cos, sin) of slots e & ~1 and e | 1
    const float cos = e & 1 ? c.z : c.x, sin = e & 1 ? c.w : c.y;
    half_t h;
    if (QUAD == 0 ? e >= 1 && e <= 6 : QUAD == 1 && e >= 2) {
      float o = (e & 1) == (QUAD == 0) ? fmaf(partner[e], sin, n[e] * cos) : fmaf(n[e], cos, partner[e] * sin);
      asm volatile("" : "+v"(o));  // rounded to fp32 first
      h = (half_t)o;
    } else {
      h = (half_t)fmaf(n[e], cos, partner[e] * sin);
      // Kept apart from its neighbour, so that the compiler fuses the rounding (v_fma_mix{lo,hi}_f16).
      if (!(e & 1)) asm volatile("" : "+v"(h));
    }
    r[e] = h;
  }
  return r;
}
__device__ inline rope_h8 rope_vector(rope_h8 x, float4 g0, float4 g1, const float4 (&c4)[4], int j, float eps, int quad) {
  float v[8], ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = (float)x[e];
    ss = fmaf(v[e], v[e], ss);
  }
  ss = row_sum(ss);
  const float inv = __frsqrt_rn(fmaf(ss, 1.0f / 128.0f, eps));
  const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
  float n[8], partner[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    n[e] = v[e] * inv * g[e];
    const float rotated = row_rotate<8>(n[e]);
    partner[e] = j < 8 ? -rotated : rotated;
  }
  return quad == 0 ? rope_rotate<0>(n, partner, c4) : quad == 1 ? rope_rotate<1>(n, partner, c4) : rope_rotate<2>(n, partner, c4);
}

constexpr int kRopeSeqs = 64;
constexpr int kRopeMaxHeads = 32;
struct RopeArgs {
  const half_t* in;       // head h < split of row t at in + t * in_stride + in_col_q + 128 h,
                          // head h >= split at in + t * in_stride + in_col_k + 128 (h - split)
  half_t* out_q;          // head h < split of row t at out_q + t * out_stride_q + 128 h
  half_t* out_k;          // head h >= split at out_k + t * out_stride_k + 128 (h - split)
  const float* weight_q;  // gains of the first `split` heads (NULL: 1)
  const float* weight_k;  // gains of the others (NULL: 1)
  const float2* rope;     // [position][64] (cos, sin), f32 of the f64 angle (model.ts:76-81)
  int64_t in_stride, out_stride_q, out_stride_k;
  int64_t in_col_q, in_col_k;
  int32_t heads, split;   // head vectors per token: 4 * ITERS; split a multiple of 4
  float eps;
  int32_t nseq;
  int32_t cu[kRopeSeqs + 1];  // token offsets of this launch's sequences (cu[0] = first token)
};

// One launch per kRopeSeqs sequences of cu (host array of nseq + 1 offsets); the rest of `a`
// filled by the caller.
hipError_t launch_qk_norm_rope(RopeArgs a, const int32_t* cu, int nseq, hipStream_t stream);

}  // namespace qattn
