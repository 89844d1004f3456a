// q4_matmul.hip -- Q4_0 "tile32-compact" dequant-GEMM: Y = X W^T with fp16 activations X [M, K]
// and 4-bit weights W [N, K]: the model's four projections (QKV, attention output, gate/up, down).
//
// Replaces the reference's compact batch matmul (src/webgpu/quant-matmul.ts:267-307, dequant
// :99-108) over the layout written by packQ40Tile32 (src/prepacked/format.ts:64-96): 20-byte
// records (f16 scale, 2 pad bytes, 16 quant bytes; element j of the 32-column block in the low
// nibble of byte j, element j+16 in its high nibble) ordered ((n/32) * (K/32) + k/32) * 32 + n%32.
// The weight is f16(scale * (q - 8)), as the reference dequantises it; the products and sums run
// in fp32 on the matrix cores (the reference accumulates in f16).
//
// Four kernels, one result: every output element is the same MFMA chains (one per 1,024 columns of K,
// its K blocks in turn from a zero accumulator; the chains' sums added in order), so a row does not
// depend on the launch it is in.  v_mfma_f32_16x16x32_f16 on a K block equals two chained
// v_mfma_f32_32x32x16_f16 on its halves bit for bit, which lets each kernel take the shape it needs.
//   * q4_tile_kernel, large launches: 256 x 256 / 256 x 128 / 128 x 128 workgroup tiles, X by
//     LDS-DMA, every weight record dequantised once per workgroup into an LDS tile;
//   * q4_mid_kernel, medium launches: 64 x 128 tiles, X by LDS-DMA, the weights dequantised
//     straight into each wavefront's MFMA fragments;
//   * q4_direct_kernel, K above 1024 and at most kQ4DirectBlocks 32 x 32 output blocks: a wavefront
//     per block, no tile staging;
//   * q4_small_kernel, the smallest launches: a workgroup per 16- or 32-row block, K shared out.
// Tiles are numbered so that consecutive workgroups on one XCD (workgroup b runs on XCD b % 8)
// walk the N tiles of one M tile: its X rows stay in that XCD's L2.  The SWIGLU variants (the FFN's
// gate/up projection, model.ts:126-127) map B rows onto a feature's gate and up rows and write
// silu(gate) * up instead of the projection.
#include <hip/hip_runtime.h>
#include <stdint.h>


#include "model_ops.h"
#include "qk_rope.h"

namespace qattn {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kQ4Record = 20;  // bytes per (row, 32-column block)
// Every output element is the fp32 sum, in order, of MFMA chains over chunks of kQ4Chunk K blocks
// (1,024 columns), each chain from a zero accumulator: y = f16((c0 + c1) + c2) for K = 3072.  The
// split depends on K alone, so a row's result does not depend on the batch, the length of a chain
// (and with it the bound of its rounding error) does not grow with K, and the chunks of a launch
// with few tiles run side by side.
constexpr int kQ4Chunk = 32;
__host__ __device__ constexpr int q4_chunks(int K) { return (K / 32 + kQ4Chunk - 1) / kQ4Chunk; }
__device__ inline __amdgpu_buffer_rsrc_t q4_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// Four weights of four quant bytes: f16(scale * (q - 8)) of their low (HIGH = false) or high
// nibbles.  A byte under 0x64 is the f16 1024 + byte; q - 8 follows exactly (for high nibbles
// 1024 + 16 q -> 64 + q - 72 in one fma), and one f16 multiply rounds as the reference's does.
template <bool HIGH>
__device__ inline u2 dequant4(uint32_t q, h2 scale) {
  const uint32_t v = q & (HIGH ? 0xF0F0F0F0u : 0x0F0F0F0Fu);
  const h2 p0 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
  const h2 p1 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
  h2 c0, c1;
  if constexpr (HIGH) {
    const h2 m = {(_Float16)0.0625f, (_Float16)0.0625f}, k = {(_Float16)-72.0f, (_Float16)-72.0f};
    c0 = __builtin_elementwise_fma(p0, m, k);
    c1 = __builtin_elementwise_fma(p1, m, k);
  } else {
    const h2 k = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    c0 = p0 + k;
    c1 = p1 + k;
  }
  return u2{__builtin_bit_cast(uint32_t, c0 * scale), __builtin_bit_cast(uint32_t, c1 * scale)};
}

// The 8 weights of a B fragment: quant bytes b0..b7 (two dwords) -> low or high nibbles.
template <bool HIGH>
__device__ inline h8 dequant8(u2 q, h2 scale) {
  const u2 a = dequant4<HIGH>(q[0], scale), b = dequant4<HIGH>(q[1], scale);
  return __builtin_bit_cast(h8, u4{a[0], a[1], b[0], b[1]});
}

// Buffer ranges.  The range check covers the per-lane offset (and the instruction's), not the scalar one
// that carries the K block, so a range ends exactly where its last row or weight tile does: w_bytes is the
// tensor's own size, and a row past M or a weight row past the last tile of 32 lies outside whatever its K
// block.  A row's K blocks lie within the row (K <= ldx).  Tiles overhang M by at most 255 rows:
// (M + 255) * ldx * 2 < 2^32 for every x that the entry points accept ((M + 128) * ldx * 2 < 2^31), so
// their offsets do not wrap.
typedef __attribute__((address_space(3))) void lds_void_t;

// LDS tiles: rows of 32 columns of fp16 (64 B per row) for X (A) and for the dequantised weights (B,
// row = output column n).  The four 16-byte chunks of row r sit at physical chunk
// c ^ ((r >> 2) & 3): 16 consecutive rows reading one logical chunk then cover all 64 banks, so
// the fragment reads (lanes 0-15 / 16-31 / ... take 16 consecutive rows) are conflict free.
__device__ inline uint32_t q4_lds_off(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4); }

// The memory and matrix builtins behind plain (non-template) device functions: hipcc's host pass
// drops a kernel template's host stub when such a builtin sits in a dependent context.
__device__ inline void q4_store_b16(_Float16 v, __amdgpu_buffer_rsrc_t rs, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), rs, off, 0, 0);
}
__device__ inline f16x q4_mfma(h8 a, h8 b, f16x c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
typedef float f4 __attribute__((ext_vector_type(4)));
__device__ inline f4 q4_mfma16(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ inline void q4_dma16(__amdgpu_buffer_rsrc_t rs, char* dst, uint32_t off, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)dst, 16, off, soff, 0, 0);
}
__device__ inline void q4_store16(u4 v, __amdgpu_buffer_rsrc_t rs, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b128(v, rs, off, 0, 0);
}
__device__ inline u4 q4_load16(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
}
__device__ inline void q4_store8(u2 v, __amdgpu_buffer_rsrc_t rs, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b64(v, rs, off, 0, 0);
}
__device__ inline uint32_t q4_pack(_Float16 a, _Float16 b) {
  return (uint32_t)__builtin_bit_cast(unsigned short, a) | (uint32_t)__builtin_bit_cast(unsigned short, b) << 16;
}

// Waits for all but the newest V vector-memory operations and for all LDS operations of this
// wavefront, then meets the workgroup.  One block of its own: the compiler's barrier would wait
// for every LDS-DMA load in flight.
template <int V>
__device__ inline void q4_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(V) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

#define Q4_INLINE __attribute__((always_inline))

// ---- large launches.
// Workgroup tile 32 MF x 64 NWN, 2 x NWN wavefronts of 16 MF x 64 per group.  K above 1024: G = 2 or 3
// such groups, one per chunk of K, whose chains meet through LDS at the end, or (FOLD) one group that
// runs the chunks in turn and adds each finished chain to a second set of accumulators.
//
// What bounds it: LDS bandwidth (128 B per clock and CU, measured) and power.  A 128 x 64 wavefront
// (MF = 8) reads 12 KiB of fragments per K block for 512 clocks of MFMA, so two per SIMD keep LDS
// busy about 1,020 of 1,024 clocks at 256 x 256 (1,150 at 256 x 128); the 64 x 64 wavefronts this
// replaces needed 1.4x the MFMA time in LDS.  16x16x32 MFMAs sustain 1.9 PFLOP/s under this card's
// power limit, 32x32x16 ones 1.65 (pure MFMA loops).  Hence the large wavefront tiles, the 16 x 16
// instruction, and the vector-memory instructions spread one per several MFMAs: issued in a burst
// after the barrier they filled the texture unit's queue and stalled the MFMAs behind them (70.5 ->
// 68.1 us).  Not kept: weights dequantised into registers at this size (VALU power: 73 us), four
// wavefronts of 128 x 128 (one per SIMD cannot issue the dequantisation beside its MFMAs: 65 us).
// The folding 128 x 256 tile spreads its loads and dequantising the same way (8000 x 3072 -> 1024 57.9 ->
// 54.1 us); its 64 x 64 wavefronts leave registers for the second set of accumulators.
// Measured (us, before -> after): 8000 x 1024 -> 4096 80.4 -> 65.5; 20000 x 1024 -> 6144 with SwiGLU
// 292 -> 254; 8000 x 2048 -> 1024 44.8 -> 38.8; 8000 x 3072 -> 1024 66.7 -> 54.1.
//
// Step kb (X tile and weight tile kb in LDS; the first half's fragments in registers): half 1 reads
// the other row fragments, dequantises weight tile kb + 1 into the free B buffer and runs the first
// half's MFMAs; the barrier publishes that tile and X tile kb + 1 (loaded two steps ago); half 2
// reads the next step's fragments under the other half's MFMAs.  X tile kb + 3 goes into the buffer
// that tile kb - 1 left at the previous barrier.
template <bool SWIGLU, int MF, int NWN, int G, bool FOLD>
__global__ __launch_bounds__(128 * NWN * G, 2) void q4_tile_kernel(
    const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N, _Float16* y, int64_t ldy,
    int tiles_n, int tiles_total, int per_xcd) {
  constexpr int kWaves = 2 * NWN;                            // per group
  constexpr int kTileM = 32 * MF, kTileN = 64 * NWN;
  constexpr int kBytesA = kTileM * 64, kBytesB = kTileN * 64;  // one K block's tiles
  constexpr int AJ = MF / NWN;                               // X loads per wavefront and K block
  constexpr int A1 = AJ / 2, A2 = AJ - A1;                   // ... in the first / second half step
  constexpr int H = MF / 2;                                  // row fragments per half step
  __shared__ __attribute__((aligned(1024))) char sA0[G * kBytesA];
  __shared__ __attribute__((aligned(1024))) char sA1[G * kBytesA];
  __shared__ __attribute__((aligned(1024))) char sA2[G * kBytesA];
  __shared__ __attribute__((aligned(1024))) char sA3[G * kBytesA];
  __shared__ __attribute__((aligned(1024))) char sB0[G * kBytesB];
  __shared__ __attribute__((aligned(1024))) char sB1[G * kBytesB];

  const int u = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (u >= tiles_total) return;
  const int m0 = (u / tiles_n) * kTileM, n0 = (u % tiles_n) * kTileN;
  const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = G == 1 ? 0 : gwave / kWaves, wave = G == 1 ? gwave : gwave % kWaves;
  const int lane = threadIdx.x & 63, tid = 64 * wave + lane;
  const int l16 = lane & 15, kq = lane >> 4;
  const int wr = 16 * MF * (wave & 1), wc = 64 * (wave >> 1);
  const int kblocks = K >> 5;
  const int kb0 = G == 1 ? 0 : grp * kQ4Chunk, kn = G == 1 ? kblocks : kQ4Chunk;
  const int k_here = min(kn, kblocks - kb0);  // blocks from k_here on are read as zeros

  const uint32_t x_bytes = (uint32_t)M * (uint32_t)ldx * 2u;
  uint32_t a_src[AJ];
#pragma unroll
  for (int j = 0; j < AJ; ++j) {
    const int row = 16 * (AJ * wave + j) + (lane >> 2);
    a_src[j] = (uint32_t)(m0 + row) * (uint32_t)ldx * 2u + 16u * ((lane & 3) ^ ((row >> 2) & 3));
  }
  const uint32_t a_dst = grp * kBytesA + 1024 * AJ * wave;
  // X loads j0 .. j0 + n - 1 of K block kb: 16 rows (1 KiB) per wavefront instruction; lane's LDS slot
  // is row lane / 4, physical chunk lane & 3.
  auto load_a = [&](char* dst, int kb, int j0, int n) Q4_INLINE {
    const auto rs = q4_rsrc(x, kb < k_here ? x_bytes : 0u);
#pragma unroll
    for (int j = j0; j < j0 + n; ++j) q4_dma16(rs, dst + a_dst + 1024 * j, a_src[j], (uint32_t)(kb0 + kb) * 64u);
  };
  // Thread (row n = tid / 2, half h = tid & 1) dequantises quant bytes 8h .. 8h + 7 of the record of
  // (n0 + n, kb): columns 8h .. + 7 (chunk h) and 16 + 8h .. + 7 (chunk 2 + h).  SWIGLU: B rows 0-31
  // of each 64 are gate rows of 32 features, rows 32-63 their up rows.
  const int brow = tid >> 1, bhalf = tid & 1;
  const int wtile = SWIGLU ? ((brow >> 5) & 1 ? N >> 6 : 0) + (n0 >> 6) + (brow >> 6) : (n0 + brow) >> 5;
  const uint32_t w_rec = ((uint32_t)wtile * (uint32_t)kblocks * 32u + (uint32_t)(brow & 31)) * kQ4Record;
  const uint32_t w_q = w_rec + 4u + 8u * bhalf;
  const uint32_t b_lo = grp * kBytesB + q4_lds_off(brow, bhalf), b_hi = grp * kBytesB + q4_lds_off(brow, 2 + bhalf);
  struct WRegs {
    uint32_t scale;
    u2 q;
  };
  auto w_rs = [&](int kb) Q4_INLINE { return q4_rsrc(w, kb < k_here ? w_bytes : 0u); };
  auto load_ws = [&](WRegs& r, int kb) Q4_INLINE {
    r.scale = __builtin_amdgcn_raw_buffer_load_b32(w_rs(kb), w_rec, (uint32_t)(kb0 + kb) * (32u * kQ4Record), 0);
  };
  auto load_wq = [&](WRegs& r, int kb) Q4_INLINE {
    r.q = __builtin_amdgcn_raw_buffer_load_b64(w_rs(kb), w_q, (uint32_t)(kb0 + kb) * (32u * kQ4Record), 0);
  };
  auto store_b = [&](char* dst, const WRegs& r) Q4_INLINE {
    const _Float16 s = __builtin_bit_cast(h2, r.scale)[0];
    const h2 scale = {s, s};
    *reinterpret_cast<h8*>(dst + b_lo) = dequant8<false>(r.q, scale);
    *reinterpret_cast<h8*>(dst + b_hi) = dequant8<true>(r.q, scale);
  };
  f4 acc[MF][4];
#pragma unroll
  for (int mb = 0; mb < MF; ++mb)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = f4{};
  const uint32_t a_rd = grp * kBytesA + q4_lds_off(wr + l16, kq), b_rd = grp * kBytesB + q4_lds_off(wc + l16, kq);

  WRegs wreg[4];
  h8 a_lo[H], a_hi[H], b0[4], b1[4];
  auto read_a = [&](h8 (&f)[H], const char* p) Q4_INLINE {
#pragma unroll
    for (int i = 0; i < H; ++i) f[i] = *reinterpret_cast<const h8*>(p + 1024 * i);
  };
  auto read_b = [&](h8 (&f)[4], const char* p) Q4_INLINE {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = *reinterpret_cast<const h8*>(p + 1024 * i);
  };
  auto mma = [&](const h8 (&b)[4], const h8 (&a)[H], int m8) Q4_INLINE {
#pragma unroll
    for (int mb = 0; mb < H; ++mb)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[m8 + mb][nb] = q4_mfma16(b[nb], a[mb], acc[m8 + mb][nb]);
  };
  load_ws(wreg[0], 0);
  load_wq(wreg[0], 0);
  load_a(sA0, 0, 0, AJ);
  __builtin_amdgcn_sched_barrier(0);
  load_ws(wreg[1], 1);
  load_a(sA1, 1, 0, AJ);
  __builtin_amdgcn_sched_barrier(0);
  load_wq(wreg[1], 1);
  load_ws(wreg[2], 2);
  load_a(sA2, 2, 0, AJ);
  __builtin_amdgcn_sched_barrier(0);
  load_wq(wreg[2], 2);
  store_b(sB0, wreg[0]);
  q4_barrier<4 + 2 * AJ>();  // X tile 0: newer are W(1), X(1), W(2), X(2)
  read_b(b0, sB0 + b_rd);
  read_a(a_lo, sA0 + a_rd);
  auto step = [&](const char* a_cur, const char* a_nxt, char* a_new, char* b_nxt, h8 (&b_cur)[4], h8 (&b_new)[4],
                  const WRegs& w_use, WRegs& w_new, int kb) Q4_INLINE {
    read_a(a_hi, a_cur + a_rd + 1024 * H);
    load_ws(w_new, kb + 3);
    load_a(a_new, kb + 3, 0, A1);
    store_b(b_nxt, w_use);
    mma(b_cur, a_lo, 0);
    if constexpr (FOLD && NWN == 4) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    if constexpr (MF == 8) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (i <= A1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
    }
    // X tile kb + 1: newer are at least step kb - 1's AJ + 2 loads and this half's 1 + A1.
    q4_barrier<3 + AJ + A1>();
    read_b(b_new, b_nxt + b_rd);
    read_a(a_lo, a_nxt + a_rd);
    load_a(a_new, kb + 3, A1, A2);
    load_wq(w_new, kb + 3);
    mma(b_cur, a_hi, H);
    if constexpr (FOLD && NWN == 4) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (j == 2) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    if constexpr (MF == 8) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (i <= A2) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (4 * i + j < 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto steps = [&](int kb) Q4_INLINE {  // blocks past the end add zero products
    step(sA0, sA1, sA3, sB1, b0, b1, wreg[1], wreg[3], kb);
    step(sA1, sA2, sA0, sB0, b1, b0, wreg[2], wreg[0], kb + 1);
    step(sA2, sA3, sA1, sB1, b0, b1, wreg[3], wreg[1], kb + 2);
    step(sA3, sA0, sA2, sB0, b1, b0, wreg[0], wreg[2], kb + 3);
  };
  if constexpr (FOLD) {
    f4 sum[MF][4];
    for (int c = 0; c < kn; c += kQ4Chunk) {
      const int end = min(c + kQ4Chunk, kn);
      for (int kb = c; kb < end; kb += 4) steps(kb);
#pragma unroll
      for (int mb = 0; mb < MF; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          sum[mb][nb] = c ? sum[mb][nb] + acc[mb][nb] : acc[mb][nb];
          acc[mb][nb] = f4{};
        }
    }
#pragma unroll
    for (int mb = 0; mb < MF; ++mb)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = sum[mb][nb];
  } else {
#pragma unroll 1
    for (int kb = 0; kb < kn; kb += 4) steps(kb);
  }
  q4_barrier<0>();

  // G > 1: the groups' chains meet.  Group g < 2 finishes the rows of half g of every wavefront's tile.
  if constexpr (G > 1) {
    char* const ex = (wave == 0 ? sA0 : wave == 1 ? sA1 : wave == 2 ? sA2 : sA3) + 16 * lane;
    auto send = [&](int m8, char* p) Q4_INLINE {
#pragma unroll
      for (int mb = 0; mb < H; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) *reinterpret_cast<f4*>(p + 1024 * (4 * mb + nb)) = acc[m8 + mb][nb];
    };
    if (grp == 0)
      send(H, ex);
    else if (G == 2 || grp == 1)
      send(0, ex + 4096 * H);
    __syncthreads();
    auto take = [&](int m8, const char* p) Q4_INLINE {
#pragma unroll
      for (int mb = 0; mb < H; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = acc[m8 + mb][nb] + *reinterpret_cast<const f4*>(p + 1024 * (4 * mb + nb));
    };
    if (grp == 0)
      take(0, ex + 4096 * H);
    else if (G == 2 || grp == 1)
      take(H, ex);
    __syncthreads();
    if constexpr (G == 3) {
      if (grp == 2) {
        send(0, ex);
        send(H, ex + 4096 * H);
      }
      __syncthreads();
      if (grp < 2) take(0, ex + 4096 * H * grp);
      __syncthreads();
      if (grp == 2) return;
    }
  }

  // Output through LDS, kRows rows of a wavefront at a time: 16 stores of 16 bytes per lane in whole
  // 128-byte lines instead of 128 stores of two bytes.  Lane (l16, kq) holds row 16 mb + l16, columns
  // 16 nb + 4 kq .. +3.
  constexpr int kMine = G > 1 ? H : MF;               // row fragments this wavefront finishes
  constexpr int kWriters = kWaves * (G > 1 ? 2 : 1);
  constexpr int kHold = 4 * G * kBytesA / 128 / kWriters;  // rows the X buffers hold for every writer
  constexpr int kMost = kHold < 64 ? kHold : 64;
  constexpr int kRows = 16 * kMine < kMost ? 16 * kMine : kMost;  // rows per pass
  constexpr int kPer = G * kBytesA / (128 * kRows);    // wavefronts per X buffer
  static_assert(4 * kPer >= kWriters && 16 * kMine % kRows == 0 && kRows % 16 == 0, "a stage per writer, whole fragments");
  const int slot = gwave / kPer;
  char* const stage = (slot == 0 ? sA0 : slot == 1 ? sA1 : slot == 2 ? sA2 : sA3) + 128 * kRows * (gwave % kPer);
  const auto yrs = q4_rsrc(y, (uint32_t)M * (uint32_t)ldy * 2u);
  const int row0 = m0 + wr + 16 * kMine * grp;
  const int n_out = SWIGLU ? N >> 1 : N;
  const int col0 = SWIGLU ? (n0 + wc) >> 1 : n0 + wc;
  constexpr int kChunks = SWIGLU ? 4 : 8;  // 16-byte pieces of a row
  auto at = [&](int row, int c) Q4_INLINE {
    return stage + row * (16 * kChunks) + ((SWIGLU ? c ^ ((row >> 2) & 3) : c ^ ((row >> 1) & 7)) << 4);
  };
#pragma unroll
  for (int p = 0; p < 16 * kMine / kRows; ++p) {
#pragma unroll
    for (int mb = 0; mb < kRows / 16; ++mb) {
      const f4(&v)[4] = acc[p * (kRows / 16) + mb];
      const int row = 16 * mb + l16;
#pragma unroll
      for (int nb = 0; nb < (SWIGLU ? 2 : 4); ++nb) {
        u2 d;
        if constexpr (SWIGLU) {  // columns 0-31: gate, 32-63: up, of the same 32 features
          const f4 &g = v[nb], &t = v[nb + 2];
          d = u2{q4_pack(swiglu_value((_Float16)g[0], (_Float16)t[0]), swiglu_value((_Float16)g[1], (_Float16)t[1])),
                 q4_pack(swiglu_value((_Float16)g[2], (_Float16)t[2]), swiglu_value((_Float16)g[3], (_Float16)t[3]))};
        } else {
          const f4& f = v[nb];
          d = u2{q4_pack((_Float16)f[0], (_Float16)f[1]), q4_pack((_Float16)f[2], (_Float16)f[3])};
        }
        *reinterpret_cast<u2*>(at(row, 2 * nb + (kq >> 1)) + 8 * (kq & 1)) = d;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    constexpr int kRowsPer = 64 / kChunks;  // rows per store instruction
#pragma unroll
    for (int i = 0; i < kRows / kRowsPer; ++i) {
      const int row = kRowsPer * i + lane / kChunks, c = lane % kChunks;
      const u4 v = *reinterpret_cast<const u4*>(at(row, c));
      const int m = row0 + kRows * p + row, n = col0 + 8 * c;
      const uint32_t off = ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u;
      q4_store16(v, yrs, m < M && n + 8 <= n_out ? off : 0x80000000u);
    }
    // A last piece of fewer than 8 columns goes element by element.
    const int part = (n_out - col0) >> 3;
    if ((n_out & 7) && n_out > col0 && part < kChunks) {
#pragma unroll 1
      for (int i = 0; i < kRows / 8; ++i) {
        const int row = 8 * i + (lane >> 3), m = row0 + kRows * p + row, n = col0 + 8 * part + (lane & 7);
        const _Float16 v = *reinterpret_cast<const _Float16*>(at(row, part) + 2 * (lane & 7));
        q4_store_b16(v, yrs, m < M && n < n_out ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u : 0x80000000u);
      }
    }
  }
}

template <bool SWIGLU, int MF, int NWN, int G, bool FOLD = false>
void launch_q4_tile(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                    _Float16* y, int64_t ldy, hipStream_t stream) {
  const int tiles_m = (M + 32 * MF - 1) / (32 * MF), tiles_n = (N + 64 * NWN - 1) / (64 * NWN);
  const int tiles = tiles_m * tiles_n, per_xcd = (tiles + 7) / 8;
  hipLaunchKernelGGL((q4_tile_kernel<SWIGLU, MF, NWN, G, FOLD>), dim3((unsigned)(8 * per_xcd)), dim3(128 * NWN * G), 0,
                     stream, x, ldx, M, K, w, w_bytes, N, y, ldy, tiles_n, tiles, per_xcd);
}

// ---- medium launches.
// 64 x 128 workgroup tiles, four wavefronts of 64 x 32 per group, each dequantising its own 32
// columns straight into MFMA fragments.  K above 1024: G = 2 or 3 groups, one per chunk of K, or FOLD as
// in q4_tile_kernel.
// What bounds it: with about one workgroup per CU, the latency of a K block.  An LDS weight tile
// puts dequantise -> LDS write -> barrier -> LDS read in every K block's chain (0.37 us per pair of
// halves); here only X goes through LDS, its barrier comes once per two blocks with loads six
// blocks ahead, and weight records are loaded four blocks ahead.  A wavefront's block is about 75
// instructions for 8 MFMAs, so VALU and MFMA issue are level.  Measured (us, before -> after):
// 1419 x 2048 -> 1024 22.2 -> 13.2, 1500 x 3072 -> 1024 31.2 -> 18.3, 500 x 1024 -> 4096 12.8 -> 9.4,
// 300 x 1024 -> 6144 with SwiGLU 12.6 -> 9.2.
// The 8 weights of a 16x16x32 B fragment from quant bytes b0..b7: mask keeps the lane's nibbles,
// mul / add take 1024 + byte to q - 8 (1, -1032 for low nibbles; 1/16, -72 for high ones).
__device__ inline h8 dequant_frag(u2 q, uint32_t mask, h2 mul, h2 add, uint32_t scale_word) {
  const _Float16 s = __builtin_bit_cast(h2, scale_word)[0];
  const h2 scale = {s, s};
  const uint32_t lo = q[0] & mask, hi = q[1] & mask;
  const h2 p0 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u));
  const h2 p1 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u));
  const h2 p2 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u));
  const h2 p3 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u));
  const h2 c0 = __builtin_elementwise_fma(p0, mul, add) * scale, c1 = __builtin_elementwise_fma(p1, mul, add) * scale;
  const h2 c2 = __builtin_elementwise_fma(p2, mul, add) * scale, c3 = __builtin_elementwise_fma(p3, mul, add) * scale;
  return __builtin_bit_cast(h8, u4{__builtin_bit_cast(uint32_t, c0), __builtin_bit_cast(uint32_t, c1),
                                   __builtin_bit_cast(uint32_t, c2), __builtin_bit_cast(uint32_t, c3)});
}
// A dword per lane whose 16-lane rows hold (s0 s1 s0 s1): s0 and s1 in every lane.
__device__ inline u2 spread_rows(uint32_t s) {
  const auto r = __builtin_amdgcn_permlane16_swap(s, s, false, false);
  return u2{r[0], r[1]};
}

template <bool SWIGLU, int G, bool FOLD>
__global__ __launch_bounds__(256 * G, 3) void q4_mid_kernel(const _Float16* x, int64_t ldx, int M, int K,
                                                            const uint8_t* w, uint32_t w_bytes, int N, _Float16* y,
                                                            int64_t ldy, int tiles_n, int tiles_total, int per_xcd) {
  constexpr int kTileM = 64, kTileN = 128, kBlock = kTileM * 64, kStage = 2 * kBlock;
  __shared__ __attribute__((aligned(1024))) char sA0[G * kStage];
  __shared__ __attribute__((aligned(1024))) char sA1[G * kStage];
  __shared__ __attribute__((aligned(1024))) char sA2[G * kStage];
  __shared__ __attribute__((aligned(1024))) char sA3[G * kStage];

  const int u = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (u >= tiles_total) return;
  const int m0 = (u / tiles_n) * kTileM, n0 = (u % tiles_n) * kTileN;
  const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = gwave >> 2, wave = gwave & 3;
  const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
  const int kblocks = K >> 5;
  const int kb0 = G == 1 ? 0 : grp * kQ4Chunk, kn = G == 1 ? kblocks : kQ4Chunk;
  const int k_here = min(kn, kblocks - kb0);  // blocks from k_here on are read as zeros

  const uint32_t x_bytes = (uint32_t)M * (uint32_t)ldx * 2u;
  const int arow = 16 * wave + (lane >> 2);
  const uint32_t a_src = (uint32_t)(m0 + arow) * (uint32_t)ldx * 2u + 16u * ((lane & 3) ^ ((arow >> 2) & 3));
  const uint32_t a_dst = grp * kStage + 1024 * wave;
  auto load_a = [&](char* dst, int kb) Q4_INLINE {  // K blocks kb, kb + 1
    const auto r0 = q4_rsrc(x, kb < k_here ? x_bytes : 0u), r1 = q4_rsrc(x, kb + 1 < k_here ? x_bytes : 0u);
    q4_dma16(r0, dst + a_dst, a_src, (uint32_t)(kb0 + kb) * 64u);
    q4_dma16(r1, dst + a_dst + kBlock, a_src, (uint32_t)(kb0 + kb + 1) * 64u);
  };
  // Fragment nb of this wavefront: columns n0 + 32 wave + 16 nb + l16 (SWIGLU: the gate / up rows
  // of features n0 / 2 + 16 wave + l16).
  const int c0 = SWIGLU ? (n0 >> 1) + 16 * wave : n0 + 32 * wave;
  const uint32_t tstride = (uint32_t)kblocks * 32u * kQ4Record;
  const uint32_t rec0 = (uint32_t)(c0 >> 5) * tstride + (uint32_t)((c0 & 31) + l16) * kQ4Record;
  const uint32_t rec1 = SWIGLU ? rec0 + (uint32_t)(N >> 6) * tstride : rec0 + 16u * kQ4Record;
  const uint32_t q_off0 = rec0 + 4u + 8u * (kq & 1), q_off1 = rec1 + 4u + 8u * (kq & 1);
  const uint32_t s_off = kq & 1 ? rec1 : rec0;
  const uint32_t mask = kq < 2 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
  const _Float16 mulc = (_Float16)(kq < 2 ? 1.0f : 0.0625f), addc = (_Float16)(kq < 2 ? -1032.0f : -72.0f);
  const h2 mul = {mulc, mulc}, add = {addc, addc};
  struct WRegs {
    uint32_t s;
    u2 q0, q1;
  };
  auto load_w = [&](WRegs& r, int kb) Q4_INLINE {
    const auto rs = q4_rsrc(w, kb < k_here ? w_bytes : 0u);
    const uint32_t so = (uint32_t)(kb0 + kb) * (32u * kQ4Record);
    r.s = __builtin_amdgcn_raw_buffer_load_b32(rs, s_off, so, 0);
    r.q0 = __builtin_amdgcn_raw_buffer_load_b64(rs, q_off0, so, 0);
    r.q1 = __builtin_amdgcn_raw_buffer_load_b64(rs, q_off1, so, 0);
  };
  f4 acc[4][2];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) acc[mb][0] = acc[mb][1] = f4{};
  const uint32_t a_rd = grp * kStage + q4_lds_off(l16, kq);
  struct Frags {
    h8 a[4], b[2];
  };
  Frags fe, fo;  // even and odd K blocks
  auto read_a = [&](Frags& f, const char* p) Q4_INLINE {
#pragma unroll
    for (int i = 0; i < 4; ++i) f.a[i] = *reinterpret_cast<const h8*>(p + a_rd + 1024 * i);
  };
  auto weights = [&](Frags& f, const WRegs& r) Q4_INLINE {
    const u2 sc = spread_rows(r.s);
    f.b[0] = dequant_frag(r.q0, mask, mul, add, sc[0]);
    f.b[1] = dequant_frag(r.q1, mask, mul, add, sc[1]);
  };
  auto mma = [&](const Frags& f) Q4_INLINE {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = q4_mfma16(f.b[nb], f.a[mb], acc[mb][nb]);
  };
  WRegs wreg[4];
  load_a(sA0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load_a(sA1, 2);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) load_w(wreg[i], i);
  __builtin_amdgcn_sched_barrier(0);
  load_a(sA2, 4);
  __builtin_amdgcn_sched_barrier(0);
  load_a(sA3, 6);
  q4_barrier<12 + 6>();  // X blocks 0, 1
  read_a(fe, sA0);
  weights(fe, wreg[0]);
  load_w(wreg[0], 4);
  __builtin_amdgcn_sched_barrier(0);
  // Stage of K blocks kb, kb + 1 in `cur`.  The X blocks of stage + 1 have landed by its barrier,
  // which also frees `cur` for stage + 4.  Vector-memory operations newer than that stage's last
  // X load at the barrier, wherever the compiler puts the weight loads within a half stage:
  //   steady state: two stages' X loads (4) and at least five blocks' weight loads (15);
  //   kb = 0 (X loaded before W0-3 by the prologue): W0-3 12, X 4-7 4, W4-5 6 = 22;
  //   kb = 2 (X 4, 5 loaded after W0-3): X 6-9 4, W4-7 12 = 16, the fewest;
  //   kb = 4: X 8-11 4, W4-9 18 = 22.
  auto stage = [&](char* cur, const char* nxt, WRegs& w1, WRegs& w2, int kb) Q4_INLINE {
    read_a(fo, cur + kBlock);
    weights(fo, w1);
    load_w(w1, kb + 5);
    mma(fe);
    q4_barrier<16>();
    load_a(cur, kb + 8);
    read_a(fe, nxt);
    weights(fe, w2);
    load_w(w2, kb + 6);
    mma(fo);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stages = [&](int kb) Q4_INLINE {  // blocks past the end add zero products
    stage(sA0, sA1, wreg[1], wreg[2], kb);
    stage(sA1, sA2, wreg[3], wreg[0], kb + 2);
    stage(sA2, sA3, wreg[1], wreg[2], kb + 4);
    stage(sA3, sA0, wreg[3], wreg[0], kb + 6);
  };
  if constexpr (FOLD) {
    f4 sum[4][2];
    for (int c = 0; c < kn; c += kQ4Chunk) {
      const int end = min(c + kQ4Chunk, kn);
      for (int kb = c; kb < end; kb += 8) stages(kb);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sum[i >> 1][i & 1] = c ? sum[i >> 1][i & 1] + acc[i >> 1][i & 1] : acc[i >> 1][i & 1];
        acc[i >> 1][i & 1] = f4{};
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i >> 1][i & 1] = sum[i >> 1][i & 1];
  } else {
#pragma unroll 1
    for (int kb = 0; kb < kn; kb += 8) stages(kb);
  }
  q4_barrier<0>();

  // G > 1: the groups' chains meet; group g < 2 finishes row fragments 2 g, 2 g + 1.
  if constexpr (G > 1) {
    char* const ex = (wave == 0 ? sA0 : wave == 1 ? sA1 : wave == 2 ? sA2 : sA3) + 16 * lane;
    if (grp == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<f4*>(ex + 1024 * i) = acc[2 + (i >> 1)][i & 1];
    } else if (G == 2 || grp == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<f4*>(ex + 4096 + 1024 * i) = acc[i >> 1][i & 1];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f4*>(ex + 8192 + 1024 * i) = acc[i >> 1][i & 1];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i >> 1][i & 1] = acc[i >> 1][i & 1] + *reinterpret_cast<const f4*>(ex + 4096 + 1024 * i);
    } else if (G == 2 || grp == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i >> 1][i & 1] = acc[2 + (i >> 1)][i & 1] + *reinterpret_cast<const f4*>(ex + 1024 * i);
    }
    if constexpr (G == 3) {
      if (grp < 2)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[i >> 1][i & 1] = acc[i >> 1][i & 1] + *reinterpret_cast<const f4*>(ex + 8192 + 4096 * grp + 1024 * i);
    }
    __syncthreads();
  }
  // Output through LDS (rows 0-31 in sA0, 32-63 in sA1), stored as whole rows of the tile.  Lane
  // (l16, kq) holds row 16 mb + l16, columns 16 nb + 4 kq .. +3 of the wavefront's 32.
  constexpr int kPieces = SWIGLU ? 8 : 16;  // 16-byte pieces of a row
  auto at = [&](int row, int c) Q4_INLINE {
    return (row < 32 ? sA0 : sA1) + (row & 31) * (16 * kPieces) + ((SWIGLU ? c ^ ((row >> 1) & 7) : c ^ (row & 15)) << 4);
  };
  constexpr int kGroups = G > 1 ? 2 : 1;  // that finish and store rows
  if (grp < kGroups)
#pragma unroll
  for (int i = 0; i < 4 / kGroups; ++i) {
    const int row = 32 * grp + 16 * i + l16;
    if constexpr (SWIGLU) {
      const f4 &g = acc[i][0], &t = acc[i][1];
      *reinterpret_cast<u2*>(at(row, 2 * wave + (kq >> 1)) + 8 * (kq & 1)) =
          u2{q4_pack(swiglu_value((_Float16)g[0], (_Float16)t[0]), swiglu_value((_Float16)g[1], (_Float16)t[1])),
             q4_pack(swiglu_value((_Float16)g[2], (_Float16)t[2]), swiglu_value((_Float16)g[3], (_Float16)t[3]))};
    } else {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const f4& f = acc[i][nb];
        *reinterpret_cast<u2*>(at(row, 4 * wave + 2 * nb + (kq >> 1)) + 8 * (kq & 1)) =
            u2{q4_pack((_Float16)f[0], (_Float16)f[1]), q4_pack((_Float16)f[2], (_Float16)f[3])};
      }
    }
  }
  __syncthreads();
  if (grp >= kGroups) return;
  const auto yrs = q4_rsrc(y, (uint32_t)M * (uint32_t)ldy * 2u);
  const int n_out = SWIGLU ? N >> 1 : N, col0 = SWIGLU ? n0 >> 1 : n0;
  constexpr int kRowsPer = 256 * kGroups / kPieces;  // rows per store of the workgroup
#pragma unroll
  for (int i = 0; i < kTileM / kRowsPer; ++i) {
    const int row = kRowsPer * i + (int)threadIdx.x / kPieces, c = threadIdx.x % kPieces;
    const int m = m0 + row, n = col0 + 8 * c;
    q4_store16(*reinterpret_cast<const u4*>(at(row, c)), yrs,
               m < M && n + 8 <= n_out ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u : 0x80000000u);
  }
  // A last piece of fewer than 8 columns goes element by element.
  const int part = (n_out - col0) >> 3;
  if ((n_out & 7) && part < kPieces) {
#pragma unroll 1
    for (int i = threadIdx.x; i < kTileM * 8; i += 256 * kGroups) {
      const int row = i >> 3, m = m0 + row, n = col0 + 8 * part + (i & 7);
      const _Float16 v = *reinterpret_cast<const _Float16*>(at(row, part) + 2 * (i & 7));
      q4_store_b16(v, yrs, m < M && n < n_out ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u : 0x80000000u);
    }
  }
}

template <bool SWIGLU, int G, bool FOLD = false>
void launch_q4_mid(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                   _Float16* y, int64_t ldy, hipStream_t stream) {
  const int tiles_m = (M + 63) / 64, tiles_n = (N + 127) / 128, tiles = tiles_m * tiles_n, per_xcd = (tiles + 7) / 8;
  hipLaunchKernelGGL((q4_mid_kernel<SWIGLU, G, FOLD>), dim3((unsigned)(8 * per_xcd)), dim3(256 * G), 0, stream, x, ldx, M,
                     K, w, w_bytes, N, y, ldy, tiles_n, tiles, per_xcd);
}

// ---- the smallest launches: one workgroup per 16 MB x 16 NB block of output (SWIGLU: 16 features),
// its wavefronts sharing K.  Wavefront p of a chain loads and dequantises K blocks NKB p .. + NKB - 1,
// all at once; then the chain runs through the wavefronts in turn, the accumulators passing from one
// to the next through LDS, so the sums are the same as in one wavefront.  C > 1 (K above 1024): the C
// chunks of K run side by side and are added in order at the end.
// What bounds it: a launch's fixed 3 us or so, one memory round trip, and P hand-overs of about 0.2 us;
// one wavefront running the whole chain dequantised 32 blocks in sequence instead.  Weight records
// come in as they lie in memory (three 1 KiB loads per four blocks, not twelve of scattered 4- and
// 8-byte pieces, whose address work alone took 2 us per CU) and are taken apart in LDS.
// Measured (us, before -> after): 15 x 1024 -> 4096 5.9 -> 4.5, 15 rows gate/up 6.6 -> 4.6,
// 50 x 2048 -> 1024 7.5 -> 4.6, 50 x 3072 -> 1024 10.4 -> 6.1.
template <bool SWIGLU, int MB, int NB, int NKB, int C>
__global__ __launch_bounds__(64 * C * kQ4Chunk / NKB) void q4_small_kernel(
    const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N, _Float16* y, int64_t ldy,
    int turns, int blocks_m) {
  __shared__ f4 hand[C][NB * MB][64];
  const int P = C > 1 ? kQ4Chunk / NKB : turns;  // wavefronts of a chain
  const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = C > 1 ? wv / P : 0, p = wv - h * P;  // chunk, turn
  const int m0 = (int)(blockIdx.x % (unsigned)blocks_m) * 16 * MB, nblk = (int)(blockIdx.x / (unsigned)blocks_m);
  const int kblocks = K >> 5;
  const int kb0 = h * kQ4Chunk + p * NKB, k_end = min(kblocks, (h + 1) * kQ4Chunk);

  const uint32_t x_bytes = (uint32_t)M * (uint32_t)ldx * 2u;
  const uint32_t x_off = (uint32_t)(m0 + l16) * (uint32_t)ldx * 2u + 16u * kq;
  const int c0 = SWIGLU ? 16 * nblk : 16 * NB * nblk;
  const uint32_t tstride = (uint32_t)kblocks * 32u * kQ4Record;
  const uint32_t rec0 = (uint32_t)(c0 >> 5) * tstride + (uint32_t)(c0 & 31) * kQ4Record;
  const uint32_t rec1 = SWIGLU ? rec0 + (uint32_t)(N >> 6) * tstride : rec0 + 16u * kQ4Record;
  const uint32_t mask = kq < 2 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
  const _Float16 mulc = (_Float16)(kq < 2 ? 1.0f : 0.0625f), addc = (_Float16)(kq < 2 ? -1032.0f : -72.0f);
  const h2 mul = {mulc, mulc}, add = {addc, addc};

  // This wavefront's weight records (16 NB rows x NKB blocks of 20 bytes) go to LDS as they lie in
  // memory, 16 bytes per lane; blocks past the chain's end are read as zeros.
  constexpr int kBytes = 320 * NB, kUnits = kBytes / 16;  // one K block's records
  constexpr int kRaw = (NKB * kBytes + 1023) / 1024;
  __shared__ __attribute__((aligned(1024))) char raw[C * kQ4Chunk / NKB][kRaw * 1024];
  const auto wrs = q4_rsrc(w, w_bytes);
  u4 piece[kRaw];
#pragma unroll
  for (int j = 0; j < kRaw; ++j) {
    const int unit = 64 * j + lane, kb = unit / kUnits, r = unit % kUnits;
    const uint32_t off = (r < 20 ? rec0 + 16u * r : rec1 + 16u * (r - 20)) + (uint32_t)(kb0 + kb) * 640u;
    piece[j] = q4_load16(wrs, kb < NKB && kb0 + kb < k_end ? off : 0x80000000u);
  }
  h8 a[NKB][MB];
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const auto xs = q4_rsrc(x, kb0 + i < k_end ? x_bytes : 0u);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      a[i][mb] = __builtin_bit_cast(
          h8, __builtin_amdgcn_raw_buffer_load_b128(xs, x_off + (uint32_t)(16 * mb) * (uint32_t)ldx * 2u,
                                                    (uint32_t)(kb0 + i) * 64u, 0));
  }
#pragma unroll
  for (int j = 0; j < kRaw; ++j) *reinterpret_cast<u4*>(raw[wv] + 1024 * j + 16 * lane) = piece[j];
  h8 b[NKB][NB];
  const char* const mine = raw[wv] + l16 * kQ4Record + 8 * (kq & 1) + 4;
  const char* const scales = raw[wv] + (l16 + (NB == 2 ? 16 * (kq & 1) : 0)) * kQ4Record;
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const uint32_t sw = *reinterpret_cast<const uint32_t*>(scales + kBytes * i);
    const u2 sc = NB == 2 ? spread_rows(sw) : u2{sw, sw};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const uint32_t* const q = reinterpret_cast<const uint32_t*>(mine + kBytes * i + 320 * nb);
      b[i][nb] = dequant_frag(u2{q[0], q[1]}, mask, mul, add, sc[nb]);
    }
  }
  f4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < NB * MB; ++i) acc[i / NB][i % NB] = f4{};
  for (int t = 0; t < P; ++t) {
    if (t == p) {
      if (t > 0)
#pragma unroll
        for (int i = 0; i < NB * MB; ++i) acc[i / NB][i % NB] = hand[h][i][lane];
#pragma unroll
      for (int i = 0; i < NKB; ++i)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = q4_mfma16(b[i][nb], a[i][mb], acc[mb][nb]);
      if (t < P - 1 || h > 0)
#pragma unroll
        for (int i = 0; i < NB * MB; ++i) hand[h][i][lane] = acc[i / NB][i % NB];
    }
    if (t < P - 1 || C > 1) __syncthreads();
  }
  if (h != 0 || p != P - 1) return;
  if constexpr (C > 1)
#pragma unroll
    for (int c = 1; c < C; ++c)
#pragma unroll
      for (int i = 0; i < NB * MB; ++i) acc[i / NB][i % NB] = acc[i / NB][i % NB] + hand[c][i][lane];

  const auto yrs = q4_rsrc(y, (uint32_t)M * (uint32_t)ldy * 2u);
  const int n_out = SWIGLU ? N >> 1 : N;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = m0 + 16 * mb + l16;
#pragma unroll
    for (int nb = 0; nb < (SWIGLU ? 1 : NB); ++nb) {
      const int n = c0 + 16 * nb + 4 * kq;
      _Float16 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = SWIGLU ? swiglu_value((_Float16)acc[mb][0][e], (_Float16)acc[mb][NB - 1][e]) : (_Float16)acc[mb][nb][e];
      const uint32_t off = m < M ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u : 0x80000000u;
      if (c0 + 32 <= n_out || n + 4 <= n_out) {
        q4_store8(u2{q4_pack(v[0], v[1]), q4_pack(v[2], v[3])}, yrs, off);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < n_out) q4_store_b16(v[e], yrs, off + 2u * e);
      }
    }
  }
}

constexpr int kQ4SmallChunks = 4;  // 16 wavefronts
template <bool SWIGLU, int MB, int NB>
void launch_q4_small(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                     _Float16* y, int64_t ldy, hipStream_t stream) {
  const int n_out = SWIGLU ? N / 2 : N, chunks = q4_chunks(K);
  const int blocks_m = (M + 16 * MB - 1) / (16 * MB), cols = SWIGLU ? 16 : 16 * NB, blocks = blocks_m * ((n_out + cols - 1) / cols);
  // K blocks per wavefront: few, so that its loads and dequantising are short, but each turn of the chain
  // costs a barrier: at K = 2048 four turns of eight blocks beat eight of four (50 rows: 5.1 against 5.4 us).
#define Q4_SMALL(NKB, C, P) \
  hipLaunchKernelGGL((q4_small_kernel<SWIGLU, MB, NB, NKB, C>), dim3((unsigned)blocks), dim3(64 * (P) * C), 0, stream, \
                     x, ldx, M, K, w, w_bytes, N, y, ldy, P, blocks_m)
  if constexpr (NB == 2) {
    if (chunks == 1) Q4_SMALL(4, 1, (K / 32 + 3) / 4);
  }
  if constexpr (MB == 1) {
    if (chunks == 2) Q4_SMALL(8, 2, 4);
    if (chunks == 3) Q4_SMALL(8, 3, 4);
    if (chunks == 4) Q4_SMALL(8, 4, 4);
  }
#undef Q4_SMALL
}

// ---- the small forward's fused projections: q4_small_kernel for K = 1024 whose workgroups normalise
// their own rows and, for QKV, apply the QK norm and RoPE to the head they hold.
// A workgroup's wavefronts first load their weight records, then RMSNorm the block's rows into LDS (a
// wavefront per row, repeated by every workgroup of the row block; workgroup 0 also writes the
// residual sum, to another buffer, since the others still read x), then run the chain as
// q4_small_kernel does.  QKV: 16 wavefronts hold the 128 columns of one head for 16 rows; the head goes
// through LDS to the 16-lane layout of rope_vector.
// What bounds the small forward is its launches: each costs 3 us or more whatever it does, and this
// takes three of eight out of every layer.  Measured (us, 28 layers, before -> after): 1 token 1,122 ->
// 875, 15 tokens 1,200 -> 1,070, 32 tokens 1,264 -> 1,175.  The rows normalised in every workgroup are
// VALU work that grows with the tokens: at 33 to 64 the separate launches are as fast (1,378 against
// 1,385 at 50), hence kFusedTokens.
template <bool QKV, int MB>
__global__ __launch_bounds__(QKV ? 1024 : 512) void q4_fused_kernel(FusedNorm n, const uint8_t* w, uint32_t w_bytes,
                                                                     int N, _Float16* y, int64_t ldy, int blocks_m,
                                                                     FusedQkv out) {
  constexpr int kBlocks = 32, P = QKV ? 4 : 8, NKB = kBlocks / P, G = QKV ? 4 : 1, W = P * G, kRows = 16 * MB;
  constexpr int kRaw = (NKB * 640 + 1023) / 1024;
  __shared__ __attribute__((aligned(1024))) char raw[W][kRaw * 1024];
  __shared__ __attribute__((aligned(1024))) char rows[kRows][2048];  // 16-byte chunk c of row r at c ^ (r & 15)
  __shared__ f4 hand[G][2 * MB][64];
  const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = wv / P, p = wv % P;
  const int m0 = (int)(blockIdx.x % (unsigned)blocks_m) * kRows, nblk = (int)(blockIdx.x / (unsigned)blocks_m);

  const int c0 = QKV ? 128 * nblk + 32 * g : 16 * nblk;
  const uint32_t rec0 = ((uint32_t)(c0 >> 5) * (kBlocks * 32u) + (uint32_t)(c0 & 31)) * kQ4Record;
  const uint32_t rec1 = rec0 + (QKV ? 16u : (uint32_t)(N >> 6) * (kBlocks * 32u)) * kQ4Record;
  const auto wrs = q4_rsrc(w, w_bytes);
  u4 piece[kRaw];
#pragma unroll
  for (int j = 0; j < kRaw; ++j) {
    const int unit = 64 * j + lane, kb = unit / 40, r = unit % 40;
    const uint32_t off = (r < 20 ? rec0 + 16u * r : rec1 + 16u * (r - 20)) + (uint32_t)(NKB * p + kb) * 640u;
    piece[j] = q4_load16(wrs, kb < NKB ? off : 0x80000000u);
  }
#pragma unroll
  for (int i = 0; i < kRows / W; ++i) {
    const int r = W * i + wv, m = m0 + r;
    const auto put = [&](int c, half8 v) { *reinterpret_cast<half8*>(rows[r] + (((c >> 3) ^ (r & 15)) << 4)) = v; };
    if (m < n.tokens) {
      const half_t* const xr = n.x + (size_t)m * 1024;
      if (n.residual)
        rmsnorm_row(xr, n.residual + (size_t)m * 1024, nblk == 0 ? n.x_out + (size_t)m * 1024 : nullptr, n.weight, put,
                    1024, n.eps, lane);
      else
        rmsnorm_row(xr, nullptr, nullptr, n.weight, put, 1024, n.eps, lane);
    } else {
      put(8 * lane, half8{});
      put(8 * lane + 512, half8{});
    }
  }
  const uint32_t mask = kq < 2 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
  const _Float16 mulc = (_Float16)(kq < 2 ? 1.0f : 0.0625f), addc = (_Float16)(kq < 2 ? -1032.0f : -72.0f);
  const h2 mul = {mulc, mulc}, add = {addc, addc};
#pragma unroll
  for (int j = 0; j < kRaw; ++j) *reinterpret_cast<u4*>(raw[wv] + 1024 * j + 16 * lane) = piece[j];
  h8 b[NKB][2];
  const char* const mine = raw[wv] + l16 * kQ4Record + 8 * (kq & 1) + 4;
  const char* const scales = raw[wv] + (l16 + 16 * (kq & 1)) * kQ4Record;
#pragma unroll
  for (int i = 0; i < NKB; ++i) {
    const u2 sc = spread_rows(*reinterpret_cast<const uint32_t*>(scales + 640 * i));
    const uint32_t* const q0 = reinterpret_cast<const uint32_t*>(mine + 640 * i);
    const uint32_t* const q1 = reinterpret_cast<const uint32_t*>(mine + 640 * i + 320);
    b[i][0] = dequant_frag(u2{q0[0], q0[1]}, mask, mul, add, sc[0]);
    b[i][1] = dequant_frag(u2{q1[0], q1[1]}, mask, mul, add, sc[1]);
  }
  __syncthreads();
  h8 a[NKB][MB];
#pragma unroll
  for (int i = 0; i < NKB; ++i)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      a[i][mb] = *reinterpret_cast<const h8*>(rows[16 * mb + l16] + (((4 * (NKB * p + i) + kq) ^ l16) << 4));
  f4 acc[MB][2];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb][0] = acc[mb][1] = f4{};
  for (int t = 0; t < P; ++t) {
    if (t == p) {
      if (t > 0)
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i) acc[i >> 1][i & 1] = hand[g][i][lane];
#pragma unroll
      for (int i = 0; i < NKB; ++i)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = q4_mfma16(b[i][nb], a[i][mb], acc[mb][nb]);
      if (t < P - 1)
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i) hand[g][i][lane] = acc[i >> 1][i & 1];
    }
    if (t < P - 1) __syncthreads();
  }
  if constexpr (!QKV) {
    if (p != P - 1) return;
    const int n_inter = N >> 1, f = c0 + 4 * kq;
    const auto yrs = q4_rsrc(y, (uint32_t)n.tokens * (uint32_t)ldy * 2u);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + 16 * mb + l16;
      _Float16 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = swiglu_value((_Float16)acc[mb][0][e], (_Float16)acc[mb][1][e]);
      q4_store8(u2{q4_pack(v[0], v[1]), q4_pack(v[2], v[3])}, yrs,
                m < n.tokens && f < n_inter ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)f) * 2u : 0x80000000u);
    }
  } else {
    // The head's 16 rows of 128 columns, chunk c of row r at c ^ r, over the weight records (read by
    // their own wavefronts before the first barrier).
    char* const tile = raw[0];
    if (p == P - 1) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const f4& v = acc[0][nb];
        *reinterpret_cast<u2*>(tile + l16 * 256 + (((4 * g + 2 * nb + (kq >> 1)) ^ l16) << 4) + 8 * (kq & 1)) =
            u2{q4_pack((_Float16)v[0], (_Float16)v[1]), q4_pack((_Float16)v[2], (_Float16)v[3])};
      }
    }
    __syncthreads();
    if (wv >= 4) return;
    // Wavefront wv: rows 4 wv .. + 3, lane (row 4 wv + lane / 16, j = lane % 16): columns 8 j .. + 7.
    const int row = 4 * wv + kq, t = m0 + row;
    const rope_h8 x = *reinterpret_cast<const rope_h8*>(tile + row * 256 + ((l16 ^ row) << 4));
    if (nblk >= 24) {
      if (t < n.tokens)
        *reinterpret_cast<rope_h8*>(out.qkv + (size_t)t * 4096 + 3072 + (nblk - 24) * 128 + 8 * l16) = x;
      return;
    }
    // Sequence of each token: the number of sequences that end at or before it.
    const int end = lane < out.nseq ? out.cu[lane + 1] : 0x7fffffff;
    int s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = __popcll(__ballot(end <= m0 + 4 * wv + i));
      s = kq == i ? c : s;
    }
    const int pos = t < n.tokens ? t - out.cu[s] : 0;
    const float* const gains = nblk < 16 ? out.weight_q : out.weight_k;
    const float4 g0 = reinterpret_cast<const float4*>(gains)[2 * l16], g1 = reinterpret_cast<const float4*>(gains)[2 * l16 + 1];
    const float4* const cs = reinterpret_cast<const float4*>(out.rope + (int64_t)pos * 64 + 8 * (l16 & 7));
    const float4 c4[4] = {cs[0], cs[1], cs[2], cs[3]};
    const rope_h8 r = rope_vector(x, g0, g1, c4, l16, out.eps, nblk >> 2);
    half_t* const dst = nblk < 16 ? out.q + (size_t)t * 2048 + nblk * 128 : out.k + (size_t)t * 1024 + (nblk - 16) * 128;
    if (t < n.tokens) *reinterpret_cast<rope_h8*>(dst + 8 * l16) = r;
  }
}

hipError_t launch_q4_norm_qkv(const FusedNorm& n, const uint8_t* w, uint32_t w_bytes, const FusedQkv& out,
                              hipStream_t stream) {
  const int blocks_m = (n.tokens + 15) / 16;
  hipLaunchKernelGGL((q4_fused_kernel<true, 1>), dim3((unsigned)(32 * blocks_m)), dim3(1024), 0, stream, n, w, w_bytes,
                     4096, nullptr, (int64_t)0, blocks_m, out);
  return hipGetLastError();
}

hipError_t launch_q4_norm_swiglu(const FusedNorm& n, const uint8_t* w, uint32_t w_bytes, int n_inter, half_t* y,
                                 int64_t ldy, hipStream_t stream) {
  const int mb = n.tokens <= 16 ? 1 : 2, blocks_m = (n.tokens + 16 * mb - 1) / (16 * mb);
  const dim3 grid((unsigned)(n_inter / 16 * blocks_m));
  if (mb == 1)
    hipLaunchKernelGGL((q4_fused_kernel<false, 1>), grid, dim3(512), 0, stream, n, w, w_bytes, 2 * n_inter, y, ldy,
                       blocks_m, FusedQkv{});
  else
    hipLaunchKernelGGL((q4_fused_kernel<false, 2>), grid, dim3(512), 0, stream, n, w, w_bytes, 2 * n_inter, y, ldy,
                       blocks_m, FusedQkv{});
  return hipGetLastError();
}

// ---- K above 1024, at most kQ4DirectBlocks 32 x 32 output blocks beyond q4_small_kernel's: one
// wavefront per block (or one per chunk of K), and no LDS tiles.  Each wavefront
// loads its own X rows and weight records straight into MFMA fragment registers, kQ4Ahead K blocks
// ahead, dequantises them with the same code and runs the same MFMA chain.
// Lane (l32, hl) holds X row m0 + l32 and weight row n0 + l32, columns 16 s + 8 hl .. +7 of the
// K block in step s.  SWIGLU: two chains, the gate rows n0 + l32 and the up rows n_inter + n0 + l32
// of the 32 output features n0 .. n0 + 31.
// A wavefront is bound by its own dequantisation VALU work (~0.08 us per K block, twice that with
// SWIGLU's two chains) and its X loads, which touch one cache line per row: one wavefront per
// workgroup spreads the blocks over as many CUs.  Up to 512 blocks (two per CU) it beats
// q4_mid_kernel (us: 500 x 2048 -> 1024 11.9 against 12.9, 250 x 3072 -> 1024 9.9 against 17.2).
constexpr int kQ4DirectBlocks = 512;
constexpr int kQ4Ahead = 8;  // K blocks in flight per wavefront (a ring of register stages)

// One workgroup per output block.  PAR: a wavefront per chunk of K; the chains meet in LDS and
// wavefront 0 adds them in order.  Otherwise one wavefront runs the chunks in turn and adds each
// finished chain to the sum (launches whose chunk wavefronts would crowd the CUs).
// PAR up to one output block per CU.  Measured at M = 15-240 for the output and down projections:
// 25-46% faster than one wavefront; with more blocks the second wavefronts share CUs and were up to
// 13% slower.
constexpr int kQ4ParallelBlocks = 256;
constexpr int kQ4ParallelChunks = 8;
template <bool SWIGLU, bool PAR>
__global__ __launch_bounds__(PAR ? 64 * kQ4ParallelChunks : 64) void q4_direct_kernel(
    const _Float16* __restrict__ x, int64_t ldx, int M, int K, const uint8_t* __restrict__ w, uint32_t w_bytes, int N,
    _Float16* __restrict__ y, int64_t ldy, int blocks_m, int blocks_total) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, hl = lane >> 5;
  const int chunk = PAR ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  // block g: the M blocks of one N block are consecutive (they share weight records in L2)
  const int g = blockIdx.x;
  if (g >= blocks_total) return;  // the whole workgroup: its barrier below stays uniform
  const int m0 = (g % blocks_m) * 32, n0 = (g / blocks_m) * 32;
  const int kblocks_all = K >> 5;
  // This wavefront's K blocks [kb0, kblocks): one chunk, or all of K.
  const int kb0 = PAR ? chunk * kQ4Chunk : 0;
  const int kblocks = PAR ? min(kb0 + kQ4Chunk, kblocks_all) : kblocks_all;
  const int n_out = SWIGLU ? N >> 1 : N;  // output columns

  const auto xrs = q4_rsrc(x, (uint32_t)M * (uint32_t)ldx * 2u);  // rows >= M read as zeros
  const auto wrs = q4_rsrc(w, w_bytes);                          // rows >= N read as zeros
  const auto yrs = q4_rsrc(y, (uint32_t)M * (uint32_t)ldy * 2u);
  const uint32_t x_row = (uint32_t)(m0 + l32) * (uint32_t)ldx * 2u + 16u * hl;
  auto w_rec = [&](int n) {
    return ((uint32_t)(n >> 5) * (uint32_t)kblocks_all * 32u + (uint32_t)(n & 31)) * kQ4Record;
  };
  const uint32_t wu_rec = SWIGLU ? w_rec(n_out + n0 + l32) : 0u;
  const uint32_t wg_rec = w_rec(n0 + l32);
  const uint32_t w_step = 32u * kQ4Record;

  struct Stage {
    h8 a[2];
    uint32_t sg, su;
    u2 qg, qu;
  };
  constexpr int kOps = SWIGLU ? 6 : 4;  // vector-memory instructions per K block
  auto load = [&](Stage& st, int kb) {
    kb = kb < kblocks ? kb : kblocks - 1;  // past the end: re-read the last block (never used)
    const uint32_t xo = x_row + (uint32_t)kb * 64u;
    st.a[0] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xrs, xo, 0, 0));
    st.a[1] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xrs, xo + 32u, 0, 0));
    const uint32_t go = wg_rec + (uint32_t)kb * w_step;
    st.sg = __builtin_amdgcn_raw_buffer_load_b32(wrs, go, 0, 0);
    st.qg = __builtin_amdgcn_raw_buffer_load_b64(wrs, go + 4u + 8u * hl, 0, 0);
    if constexpr (SWIGLU) {
      const uint32_t uo = wu_rec + (uint32_t)kb * w_step;
      st.su = __builtin_amdgcn_raw_buffer_load_b32(wrs, uo, 0, 0);
      st.qu = __builtin_amdgcn_raw_buffer_load_b64(wrs, uo + 4u + 8u * hl, 0, 0);
    }
  };
  f16x acc_g = {}, acc_u = {};
  auto mma = [&](const Stage& st) {
    const _Float16 sg = __builtin_bit_cast(h2, st.sg)[0];
    const h2 scale_g = {sg, sg};
    acc_g = q4_mfma(st.a[0], dequant8<false>(st.qg, scale_g), acc_g);
    acc_g = q4_mfma(st.a[1], dequant8<true>(st.qg, scale_g), acc_g);
    if constexpr (SWIGLU) {
      const _Float16 su = __builtin_bit_cast(h2, st.su)[0];
      const h2 scale_u = {su, su};
      acc_u = q4_mfma(st.a[0], dequant8<false>(st.qu, scale_u), acc_u);
      acc_u = q4_mfma(st.a[1], dequant8<true>(st.qu, scale_u), acc_u);
    }
  };
  Stage ring[kQ4Ahead];
  // The waits count loads in issue order: the compiler must not move them across blocks.
#pragma unroll
  for (int j = 0; j < kQ4Ahead; ++j) {
    load(ring[j], kb0 + j);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Block kb sits in stage kb % kQ4Ahead; the loads of the kQ4Ahead - 1 blocks after it may still
  // be in flight when it is used (loads retire in issue order), then its stage takes block
  // kb + kQ4Ahead.
  constexpr int kWait = (kQ4Ahead - 1) * kOps;
  static_assert(kWait < 64, "vmcnt is 6 bits");
  static_assert(kQ4Chunk % kQ4Ahead == 0, "chunks end between ring passes");
  f16x tot_g = {}, tot_u = {};
  for (int kb = kb0; kb < kblocks; kb += kQ4Ahead) {
#pragma unroll
    for (int j = 0; j < kQ4Ahead; ++j) {
      __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8) | (kWait & 15) | ((kWait >> 4) << 14));
      if (kb + j < kblocks) mma(ring[j]);
      __builtin_amdgcn_sched_barrier(0);
      load(ring[j], kb + j + kQ4Ahead);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!PAR) {
      // End of a chunk: add the chain to the sum and start the next from zero.
      if ((kb + kQ4Ahead) % kQ4Chunk == 0 || kb + kQ4Ahead >= kblocks) {
        tot_g = kb < kQ4Chunk ? acc_g : tot_g + acc_g;
        acc_g = f16x{};
        if constexpr (SWIGLU) {
          tot_u = kb < kQ4Chunk ? acc_u : tot_u + acc_u;
          acc_u = f16x{};
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  if constexpr (!PAR) {
    acc_g = tot_g;
    acc_u = tot_u;
  }
  if constexpr (PAR) {
    __shared__ f16x part_g[kQ4ParallelChunks - 1][64];
    __shared__ f16x part_u[SWIGLU ? kQ4ParallelChunks - 1 : 1][SWIGLU ? 64 : 1];
    if (chunk > 0) {
      part_g[chunk - 1][lane] = acc_g;
      if constexpr (SWIGLU) part_u[chunk - 1][lane] = acc_u;
    }
    __syncthreads();
    if (chunk > 0) return;
    for (int c = 1; kQ4Chunk * c < kblocks_all; ++c) {
      acc_g = acc_g + part_g[c - 1][lane];
      if constexpr (SWIGLU) acc_u = acc_u + part_u[c - 1][lane];
    }
  }

  // D (32 x 32): lane holds column l32 and rows 8 (r / 4) + 4 hl + r % 4.
  const int n = n0 + l32;
  if (n >= n_out) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + 8 * (r >> 2) + 4 * hl + (r & 3);
    const uint32_t off = m < M ? ((uint32_t)m * (uint32_t)ldy + (uint32_t)n) * 2u : 0x80000000u;
    if constexpr (SWIGLU)
      q4_store_b16(swiglu_value((_Float16)acc_g[r], (_Float16)acc_u[r]), yrs, off);
    else
      q4_store_b16((_Float16)acc_g[r], yrs, off);
  }
}

template <bool SWIGLU>
void launch_q4_direct(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                      _Float16* y, int64_t ldy, hipStream_t stream) {
  const int n_out = SWIGLU ? N / 2 : N;
  const int blocks_m = (M + 31) / 32, blocks = blocks_m * ((n_out + 31) / 32);
  const int chunks = q4_chunks(K);
  if (blocks <= kQ4ParallelBlocks && chunks <= kQ4ParallelChunks)
    hipLaunchKernelGGL((q4_direct_kernel<SWIGLU, true>), dim3((unsigned)blocks), dim3(64 * chunks), 0, stream, x, ldx, M,
                       K, w, w_bytes, N, y, ldy, blocks_m, blocks);
  else
    hipLaunchKernelGGL((q4_direct_kernel<SWIGLU, false>), dim3((unsigned)blocks), dim3(64), 0, stream, x, ldx, M, K, w,
                       w_bytes, N, y, ldy, blocks_m, blocks);
}

// The kernel and tile by the number of tiles, i.e. by how a launch fills the 256 CUs (times in us).
// K up to 1024:
//   * q4_small_kernel while its 16-row blocks are at most one per CU, with 32-row blocks while those are
//     at most two (N = 4096: M = 50 5.2, mid 8.5; M = 100 7.3 against 8.6);
//   * up to 512 tiles of 64 x 128: q4_mid_kernel (N = 4096: M = 1,000 14.7, 256 x 128 tiles 17.0;
//     M = 1,500, 768 tiles, 19.6 against 18.1).  It works in passes of eight K blocks, so for K up to 256 only
//     up to 256 tiles, and 128 x 128 tiles beyond (N = 1024, K = 64, M = 3,000 5.2 against 6.8), also in
//     place of 256 x 128 ones that fill a gap (M = 20,000 14.2 against 15.6);
//   * beyond, the rows a tile pads count: up to 64 rows stay with q4_mid_kernel (N = 70,016: M = 64 18.8,
//     256 x 128 tiles 37.6), and 128 x 128 tiles serve where they pad at least a quarter fewer rows, up to
//     128 and 257 to 384 (M = 100 26.8 against 39.0, M = 300 65 against 76; M = 500, 640 against 768 rows,
//     86 against 77), unless 256 x 128 tiles fit in one round, of one per CU or of two where 128 x 128 ones do
//     not (M = 300: N = 16,000 18.8 against 19.5, N = 24,000 26.9 against 27.7);
//   * then 256 x 128 tiles while they are at most one per CU (N = 6144: M = 1,000 18.2, 256 x 256
//     tiles 26.5);
//   * then 256 x 256 tiles where their last round of 256 is mostly full (N = 4096: M = 2,400 27.5
//     against 29.5, M = 8,000 65 against 68), else 256 x 128 tiles, whose second workgroup per CU
//     fills the gap (N = 6144, M = 4,000: 1.5 rounds, 60 against 53).
// K above 1024 (N = 1024):
//   * q4_small_kernel while its 16 x 16 blocks are at most one per CU (K = 2048, M = 50 4.6, 16 x 32 blocks
//     5.1; K = 3072 6.2 against 7.0), then while its 16 x 32 blocks are (K = 3072, M = 100 7.2, direct 10.5;
//     M = 150, 320 blocks, 12.2 against 10.7) and a workgroup holds a wavefront for every part of K;
//   * q4_direct_kernel up to kQ4DirectBlocks (K = 3072, M = 500 16.5, mid 17.5);
//   * up to 256 tiles of 64 x 128: q4_mid_kernel, a group per chunk (K = 2048, M = 1,419 13.2, 128 x 128
//     tiles 19.8; K = 3072 18.4);
//   * up to 128 rows and beyond 256 tiles of 128 x 128, folding q4_mid_kernel (N = 40,000, M = 100:
//     K = 2048 33.2, 128 x 128 tiles 38.9; K = 3072 47.6 against 50.6);
//   * K up to 2048: 128 x 128 tiles while at most one per CU (M = 2,400 20.3, mid 25.4, 256 x 128 27.6),
//     then 256 x 128 or 128 x 128 tiles by the rounds each needs (M = 8,000: one round of 38.8 against two
//     of 22.7);
//   * K up to 3072: 128 x 128 tiles with three groups while at most one per CU (M = 4,000 31.9; mid 37.1,
//     128 x 256 folding 49.5); beyond, three groups of larger tiles do not fit in LDS;
//   * groups run as long as a whole chunk, so where the last chunk is at most half full the chunks are folded
//     instead (K = 1536: M = 1,419 12.5 against 13.6, M = 8,000 33.7 against 36.9; K = 1792, M = 5,000 30.2
//     against 29.5), and so is K above 3072: folding q4_mid_kernel up to 512 tiles, two workgroups per CU
//     (K = 4096, M = 4,000 47.2, 128 x 256 tiles 64.4; M = 5,000, 632 tiles, 66.1 against 64.8);
//   * the rest folds the chunks in 128 x 256 tiles where their last round of 256 is mostly full (K = 3072,
//     M = 8,000 54 against 61 with 128 x 128 tiles, M = 16,000 109 against 120), else in 128 x 128 tiles, whose
//     second workgroup per CU fills the gap (M = 12,000, 1.5 rounds, 92 against 106; K = 1792 57 against 68
//     with two groups, which at K = 2048, both chunks full, take the same 66).
template <bool SWIGLU>
hipError_t launch_q4(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                     _Float16* y, int64_t ldy, hipStream_t stream) {
  const int n_out = SWIGLU ? N / 2 : N, chunks = q4_chunks(K);
  const auto tiles = [&](int tm, int tn) { return (int64_t)((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  const auto padded = [&](int tm) { return (int64_t)((M + tm - 1) / tm) * tm; };
  const auto rounds = [](int64_t t) { return (t + 255) / 256; };
#define Q4_TILE(...) launch_q4_tile<SWIGLU, __VA_ARGS__>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream)
#define Q4_MID(...) launch_q4_mid<SWIGLU, __VA_ARGS__>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream)
  if (chunks == 1) {
    const int64_t t = tiles(256, 256);
    const bool partial = t > 256 && 256 * rounds(t) * 100 > 115 * t, shallow = K <= 256;
    if (tiles(16, 32) <= 256)
      launch_q4_small<SWIGLU, 1, 2>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
    else if (tiles(32, 32) <= 512)
      launch_q4_small<SWIGLU, 2, 2>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
    else if (tiles(64, 128) <= (shallow ? 256 : 512) || M <= 64)
      Q4_MID(1);
    else if (shallow && (tiles(64, 128) <= 512 || partial))
      Q4_TILE(4, 2, 1);
    else if (4 * padded(128) <= 3 * padded(256) && tiles(256, 128) > 256 &&
             (tiles(128, 128) <= 512 || tiles(256, 128) > 512))
      Q4_TILE(4, 2, 1);
    else if (tiles(256, 128) <= 256 || partial)
      Q4_TILE(8, 2, 1);
    else
      Q4_TILE(8, 4, 1);
  } else {
    const bool fold = chunks > 3 || K - 32 * kQ4Chunk * (chunks - 1) <= 512;
    const int64_t big = rounds(tiles(256, 128)), small = rounds(tiles(128, 128)), wide = tiles(128, 256);
    if (tiles(16, 16) <= 256 && chunks <= kQ4SmallChunks && !SWIGLU)
      launch_q4_small<SWIGLU, 1, SWIGLU ? 2 : 1>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
    else if (tiles(16, 32) <= 256 && chunks <= kQ4SmallChunks)
      launch_q4_small<SWIGLU, 1, 2>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
    else if ((int64_t)((M + 31) / 32) * ((n_out + 31) / 32) <= kQ4DirectBlocks)
      launch_q4_direct<SWIGLU>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
    else if (!fold && chunks == 2 && tiles(64, 128) <= 256)
      Q4_MID(2);
    else if (!fold && tiles(64, 128) <= 256)
      Q4_MID(3);
    else if (M <= 128 && small > 1)
      Q4_MID(1, true);
    else if (!fold && chunks == 3 && small == 1)
      Q4_TILE(4, 2, 3);
    else if (fold && tiles(64, 128) <= 512)
      Q4_MID(1, true);
    else if (K != 64 * kQ4Chunk && wide > 256 && 256 * rounds(wide) * 100 > 115 * wide)
      Q4_TILE(4, 2, 1, true);
    else if (fold || chunks == 3)
      Q4_TILE(4, 4, 1, true);
    else if (small > 1 && 5 * big <= 3 * small)
      Q4_TILE(8, 2, 2);
    else
      Q4_TILE(4, 2, 2);
  }
#undef Q4_MID
#undef Q4_TILE
  return hipGetLastError();
}

hipError_t launch_q4_matmul(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes, int N,
                            _Float16* y, int64_t ldy, hipStream_t stream) {
  if (M <= 0 || N <= 0) return hipSuccess;
  return launch_q4<false>(x, ldx, M, K, w, w_bytes, N, y, ldy, stream);
}

// y [M, n_inter] = swiglu of the [gate | up] projection; the weight has 2 n_inter rows and
// n_inter is a multiple of 64.
hipError_t launch_q4_matmul_swiglu(const _Float16* x, int64_t ldx, int M, int K, const uint8_t* w, uint32_t w_bytes,
                                   int n_inter, _Float16* y, int64_t ldy, hipStream_t stream) {
  if (M <= 0 || n_inter <= 0) return hipSuccess;
  return launch_q4<true>(x, ldx, M, K, w, w_bytes, 2 * n_inter, y, ldy, stream);
}

}  // namespace qattn
