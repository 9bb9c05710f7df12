// Q4_K prefill GEMM for gfx950: C[M,N] = alpha * A[M,K] . dequant(W)[N,K]^T for M >= 16, and
// the fused gate/up projection with gated activation, on the matrix cores.
//
// Two kernels.  Both take the activations packed once per product by a pre-pass (pack_a_row_kernel / pack_a_kernel): each row
// scaled by the power of two that puts its largest element at 2^14, rounded to f16, k-permuted (packed_place: the order in which a
// dword of nibbles comes out; a contraction index may be permuted freely when both operands agree), rows zero-padded to a
// multiple of 64.  The K loops copy them as they are, and the epilogue divides the row factor out again, exactly: activations
// beyond the f16 range (65504) neither overflow nor lose small rows to subnormals.  And both rebuild weights as f16 from the
// nibbles with magic numbers ((w & 0x000F000F) | 0x64006400 is the pair (1024 + q) in f16), a packed subtract and a packed
// fma with (d * sc, -dmin * mn).
//
// q4k_wide_kernel (large products).  Tiles of up to 256 x 256 (eight waves, 128 x 64 each).  Packed activations and the raw
// super-blocks go from memory straight into LDS (gemm_wide.h's fetches: 64 k of activations in two buffers, 256 k of weights in
// two); a wave reads its fragments of the activations, and of the weights the 16 nibble bytes a lane needs for 64 k, and
// dequantises them in registers, between the matrix-core instructions of the slice before.  So a weight costs 0.56 bytes of LDS
// traffic instead of two written and two read, at the price of one dequantisation for each wave along M (two): what bounds it is
// instruction issue (154 vector instructions for 16 or 32 matrix-core ones; the matrix cores are busy 60 % of the time at 2048
// rows).  One barrier per 64 k.  Against the other kernel in tiles of its own, weights from memory, 2048 rows: 6144 x 4096 159 -> 124 us,
// 4096 x 4096 96 -> 95, 4096 x 12288 257 -> 261, gated pair 12288 x 4096 423 -> 400; 512 rows: 64 -> 57, 58 -> 42, 149 -> 83, 152 -> 118.
// Tried there: four activation buffers instead of two (no change: a fetch is not what a step waits for), the weights
// dequantised to f16 in memory by a pre-pass for gemm_wide.h (the same at 2048 rows, slower below).
//
// Products of few rows take it too, on tiles of 32 or 64 rows whose waves share k (choose_narrow).
//
// q4k_gemm_kernel (the rest): a wave computes a 64 x 64 (or 32 x 32) quadrant with v_mfma_f32_32x32x16_f16, four waves a
// 128 x 128 (64 x 64) tile, and a workgroup is one or two such groups stacked along M against the same weight tile.  K advances 64
// at a time; a thread loads 8 or 16 nibble bytes of a row and the block header, and the weights of a tile are dequantised once
// per workgroup into LDS.  Both tiles sit in LDS as [row][64 k] with a 16-byte pad (conflict-free 16-byte fragment reads) and are
// double-buffered, one barrier per K step.
// Its K loop is bound by instruction issue, not by memory and not by the matrix cores alone.  Measured on this part: a wave issues an
// independent vector instruction every 5 cycles and a dependent one every 8, a matrix-core instruction occupies its pipe for 32.  Hence:
//   * every wave both multiplies and produces, and the producer's work of a step (LDS stores of the A tile, scale unpack,
//     nibble dwords, the loads two tiles ahead) is dealt out in pieces behind the matrix-core instructions of the same step,
//     in program order pinned with scheduling barriers;
//   * fragments are double-buffered in registers, so LDS latency runs under the previous slice;
//   * all global loads are unconditional: one conditional load makes the compiler wait for every outstanding load before a
//     tile is used, which halves the lookahead.
// Tried there and measured slower: producer / multiplier wave specialisation, two A sub-tiles per wave, 256 x 64 blocks.
#include <algorithm>
#include <cstdlib>

#include "gemm_wide.h"
#include "q4k_device.h"

namespace {

using dh::kBlockBytes;
using dh::kQK;

typedef __attribute__((ext_vector_type(8))) _Float16 half8_t;
typedef __attribute__((ext_vector_type(2))) _Float16 half2_t;
typedef __attribute__((ext_vector_type(16))) float float16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

int env_ksplit() { return dh::tuning_int("DH_GEMM_KSPLIT", 0); }

constexpr int BK = 64;
constexpr int LDS_ROW = BK + 8;                    // halves per LDS row (144 bytes)

struct GemmArgs {
  const float* A;        // [M][K]
  const _Float16* Apk;   // [M][kpad] packed activations (see pack_a_kernel)
  int kpad;              // K rounded up to a multiple of 64
  const uint8_t* W;      // Q4_K rows [N][nb*144]
  const uint8_t* W2;     // second matrix (DUAL) or null
  void* C;               // [M][N] f32 or f16
  const float* residual; // [M][N] or null
  int M, N, K, nb;
  float alpha;
  int c_f16, activation;
  float clamp_max;
  // split-K: blockIdx.z takes K steps [z * kt_per_split, ...) and writes its raw partial product to
  // partial[z][M][N]; splitk_reduce_kernel adds the pieces in order
  int ksplit, kt_per_split;
  float* partial;
  int tiles_m, tiles_n;
  const float2* row_scale;   // [M] (multiplier applied before the f16 rounding, its inverse)
  // RMSNorm prologue (norm_weight null = off): rows are normalised while they are packed
  const float* norm_weight;  // [K]
  float norm_eps;
  int norm_weight_offset;    // 1: scale by (1 + w)
};

// Where k .. k + 3 (k a multiple of 4) of a packed row lie: inside every 64, the 16 a matrix-core instruction contracts are, for either half
// h of the wave, four low nibbles' k = 16 h + 4 i .. and the four high nibbles' 32 + 16 h + 4 i .. of one dword of a weight row.
__device__ __forceinline__ int packed_place(int k) {
  const int q = k >> 2;
  return (k & ~63) + 16 * (q & 3) + 8 * ((q >> 2) & 1) + 4 * ((q >> 3) & 1);
}

// Packs the activations for the matrix cores, one wave per row (four rows per workgroup):
// finds the row's largest magnitude, scales by the power of two that puts it at 2^14 ((1, 1) for
// an all-zero row), rounds to f16 and writes the row with its k in (0, 2, 1, 3) order inside
// every group of four (the order the masked nibble pairs of the weights come out in), zero-padded
// to kpad.  out_scale[m] = (factor, 1 / factor).
__global__ __launch_bounds__(256) void pack_a_kernel(const float* __restrict__ A, int M, int K, int kpad,
                                                     _Float16* __restrict__ Apk, float2* __restrict__ out_scale) {
  const int lane = threadIdx.x & 63, m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const float* row = A + (int64_t)m * K;
  const bool vec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  float mx = 0.f;
  if (vec) {
    for (int k = 4 * lane; k < K; k += 256) {
      const float4 v = *reinterpret_cast<const float4*>(row + k);
      mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
  } else {
    for (int k = lane; k < K; k += 64) mx = fmaxf(mx, fabsf(row[k]));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  int e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
  e = max(-100, min(100, e));
  if (!(mx > 0.f) || !(mx < INFINITY)) e = 14;
  const float mul = __uint_as_float((uint32_t)(127 + 14 - e) << 23);
  if (lane == 0) out_scale[m] = make_float2(mul, __uint_as_float((uint32_t)(127 - 14 + e) << 23));
  _Float16* dst = Apk + (int64_t)m * kpad;
  for (int k = 4 * lane; k < kpad; k += 256) {
    float v[4];
    if (vec && k + 3 < K) {
      const float4 t = *reinterpret_cast<const float4*>(row + k);      // second read: cache hit
      v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = k + j < K ? row[k + j] : 0.f;
    }
    const half2_t p0 = {(_Float16)(v[0] * mul), (_Float16)(v[2] * mul)};
    const half2_t p1 = {(_Float16)(v[1] * mul), (_Float16)(v[3] * mul)};
    *reinterpret_cast<uint2*>(dst + packed_place(k)) = make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
  }
}

// The same packing with one workgroup per row and the row held in registers (NV float4 per
// thread, K <= 4 THREADS NV): every load of a row is in flight at once and the row is read once.  One
// wave per row walks its row in dependent steps and is latency-bound (14.5 us for 512 x 6912).  Rows beyond 8192 elements have
// sixteen waves: what a thread does for its sixteen pieces one after the other is the chain of a launch of few rows, and their registers leave
// one workgroup of many to a compute unit (us, 256 / 1024 threads: 47 x 8704 5.6 / 4.1, 300 x 12288 7.4 / 6.2, 2048 x 12288 36.8 / 26.3, which
// is 5.7 TB/s; but 512 x 6912 5.5 / 5.8, and 6.0 with 512).
template <int NV, int THREADS>
__global__ __launch_bounds__(THREADS) void pack_a_row_kernel(const float* __restrict__ A, int M, int K, int kpad,
                                                         _Float16* __restrict__ Apk, float2* __restrict__ out_scale,
                                                         const float* __restrict__ norm_w, float norm_eps,
                                                         int norm_w_offset) {
  constexpr int WAVES = THREADS / 64;
  __shared__ float wave_max[WAVES];
  __shared__ float wave_ss[WAVES];
  const int tid = threadIdx.x, m = blockIdx.x;
  const float* row = A + (int64_t)m * K;
  const bool vec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  float v[NV][4];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int k = 4 * tid + 4 * THREADS * i;
    if (vec && k + 3 < K) {
      const float4 t = *reinterpret_cast<const float4*>(row + k);
      v[i][0] = t.x; v[i][1] = t.y; v[i][2] = t.z; v[i][3] = t.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) v[i][j] = k + j < K ? row[k + j] : 0.f;
    }
  }
  if (norm_w) {
    // RMSNorm of the row, same arithmetic as the stand-alone kernel: x * rsqrt(mean x^2 + eps) * w
    float wn[NV][4];
    const bool wvec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(norm_w) & 15) == 0;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int k = 4 * tid + 4 * THREADS * i;
      if (wvec && k + 3 < K) {
        const float4 t = *reinterpret_cast<const float4*>(norm_w + k);
        wn[i][0] = t.x; wn[i][1] = t.y; wn[i][2] = t.z; wn[i][3] = t.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) wn[i][j] = k + j < K ? norm_w[k + j] : 0.f;
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) ss = fmaf(v[i][j], v[i][j], ss);
    ss = dh::group_combine<1, 64>(ss, dh::AddOp{});
    if ((tid & 63) == 0) wave_ss[tid >> 6] = ss;
    __syncthreads();
    float total = wave_ss[0];
#pragma unroll
    for (int w = 1; w < WAVES; w++) total += wave_ss[w];
    const float inv = 1.0f / sqrtf(total / (float)K + norm_eps);
#pragma unroll
    for (int i = 0; i < NV; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) v[i][j] = v[i][j] * inv * (norm_w_offset ? 1.0f + wn[i][j] : wn[i][j]);
  }
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) mx = fmaxf(mx, fabsf(v[i][j]));
  mx = dh::group_combine<1, 64>(mx, dh::MaxOp{});
  if ((tid & 63) == 0) wave_max[tid >> 6] = mx;
  __syncthreads();
  mx = wave_max[0];
#pragma unroll
  for (int w = 1; w < WAVES; w++) mx = fmaxf(mx, wave_max[w]);
  int e = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
  e = max(-100, min(100, e));
  if (!(mx > 0.f) || !(mx < INFINITY)) e = 14;
  const float mul = __uint_as_float((uint32_t)(127 + 14 - e) << 23);
  if (tid == 0) out_scale[m] = make_float2(mul, __uint_as_float((uint32_t)(127 - 14 + e) << 23));
  _Float16* dst = Apk + (int64_t)m * kpad;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int k = 4 * tid + 4 * THREADS * i;
    if (k < kpad) {
      const half2_t p0 = {(_Float16)(v[i][0] * mul), (_Float16)(v[i][2] * mul)};
      const half2_t p1 = {(_Float16)(v[i][1] * mul), (_Float16)(v[i][3] * mul)};
      *reinterpret_cast<uint2*>(dst + packed_place(k)) = make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
    }
  }
}

// Dequantisation in pieces, for the K loop that spreads it between the matrix-core
// instructions.  Scales of sub-blocks 2c, 2c+1 as broadcastable f16 pairs, without a branch on c:
struct PairScales {
  half2_t slo, mlo, shi, mhi;     // (scale, scale), (-min, -min) of the low- and high-nibble sub-block
};
struct ScaleBits {
  uint32_t sc, mn;                // 6-bit scales and mins of the low (byte 0) and high (byte 1) sub-block
};
__device__ __forceinline__ ScaleBits scale_bits(const u32x4_t hdr, const int c) {
  const int sh = (c & 1) * 16;
  const uint32_t a1 = hdr[1] >> sh, a2 = hdr[2] >> sh, a3 = hdr[3] >> sh;
  const bool low = c < 2;
  return ScaleBits{low ? (a1 & 0x3F3Fu) : ((a3 & 0x0F0Fu) | ((a1 >> 2) & 0x3030u)),
                   low ? (a2 & 0x3F3Fu) : (((a3 >> 4) & 0x0F0Fu) | ((a2 >> 2) & 0x3030u))};
}
__device__ __forceinline__ PairScales pair_scales_f16(const u32x4_t hdr, const ScaleBits b) {
  const float d = f16lo(hdr[0]), dmin = f16hi(hdr[0]);
  const _Float16 sl = (_Float16)(d * (float)(b.sc & 0xFFu)), sh = (_Float16)(d * (float)((b.sc >> 8) & 0xFFu));
  const _Float16 ml = (_Float16)(-dmin * (float)(b.mn & 0xFFu)), mh = (_Float16)(-dmin * (float)((b.mn >> 8) & 0xFFu));
  return PairScales{half2_t{sl, sl}, half2_t{ml, ml}, half2_t{sh, sh}, half2_t{mh, mh}};
}
// One dword of nibbles (8 weights) -> two f16 pairs of low nibbles, two of high ones.  Bits 0..3 of a half under the exponent of 1024 are
// 1024 + q, bits 4..7 under that of 64 are 64 + q: no shift brings the high nibbles down.
// The magic numbers are held in vector registers: with the constants visible the compiler emits v_and + v_or, since one instruction may
// read only one literal or scalar.
__device__ __forceinline__ uint32_t magic_number(uint32_t value) {
  uint32_t m;
  asm("v_mov_b32 %0, %1" : "=v"(m) : "i"(value));
  return m;
}
struct Magic {
  uint32_t low, high;
};
__device__ __forceinline__ Magic magic_numbers() { return Magic{magic_number(0x64006400u), magic_number(0x54005400u)}; }
__device__ __forceinline__ void dequant_low(const uint32_t w, const PairScales& ps, const Magic& m, uint32_t& p0, uint32_t& p1) {
  const half2_t k = {(_Float16)1024.f, (_Float16)1024.f};
  const half2_t v0 = __builtin_bit_cast(half2_t, (w & 0x000F000Fu) | m.low) - k;
  const half2_t v1 = __builtin_bit_cast(half2_t, ((w >> 8) & 0x000F000Fu) | m.low) - k;
  p0 = __builtin_bit_cast(uint32_t, v0 * ps.slo + ps.mlo);
  p1 = __builtin_bit_cast(uint32_t, v1 * ps.slo + ps.mlo);
}
__device__ __forceinline__ void dequant_high(const uint32_t w, const PairScales& ps, const Magic& m, uint32_t& p0, uint32_t& p1) {
  const half2_t k = {(_Float16)64.f, (_Float16)64.f};
  const half2_t v0 = __builtin_bit_cast(half2_t, (w & 0x00F000F0u) | m.high) - k;
  const half2_t v1 = __builtin_bit_cast(half2_t, ((w >> 8) & 0x00F000F0u) | m.high) - k;
  p0 = __builtin_bit_cast(uint32_t, v0 * ps.shi + ps.mhi);
  p1 = __builtin_bit_cast(uint32_t, v1 * ps.shi + ps.mhi);
}

// tanh-form GELU with tanh(t) = 1 - 2 / (1 + e^{2t}): a handful of instructions, inlined once per
// accumulator element in the epilogue.
__device__ __forceinline__ float gelu_tanh_fast(float x) {
  const float t = fminf(fmaxf(0.7978845608f * (x + 0.044715f * x * x * x), -15.0f), 15.0f);
  return 0.5f * x * (2.0f - 2.0f / (1.0f + __expf(2.0f * t)));
}


// A wave's 32 x 32 accumulator tiles: value(q, matrix, e), row(q, e) of the workgroup's tile, column col(q), a row's factor unscale(row).  A tile's
// values are computed before they are stored, and several tiles' residuals requested in front of their first store: a load behind a store waits
// for the store's trip to memory as well (sixteen of them a tile took half of 64 x 4096 x 4096 with a residual).
template <bool DUAL, int TILES, class Value, class Row, class Col, class Unscale>
__device__ __forceinline__ void store_results(const GemmArgs& a, int m0, Value&& value, Row&& row, Col&& col, Unscale&& unscale) {
  constexpr int kBatch = TILES > 4 ? 2 : TILES;         // (eight tiles leave registers for two more)
  const bool with_residual = !DUAL && a.residual && a.ksplit <= 1;
#pragma unroll
  for (int q0 = 0; q0 < TILES; q0 += kBatch) {
    float res[kBatch][16];
    if (with_residual) {
#pragma unroll
      for (int u = 0; u < kBatch; u++)
#pragma unroll
        for (int e = 0; e < 16; e++) res[u][e] = a.residual[(int64_t)min(m0 + row(q0 + u, e), a.M - 1) * a.N + min(col(q0 + u), a.N - 1)];
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      const int q = q0 + u, n = col(q);
      float v[16];
      if constexpr (DUAL) {
        auto gated = [&](auto&& act) {
#pragma unroll
          for (int e = 0; e < 16; e++) {
            const float factor = unscale(row(q, e));
            v[e] = act(value(q, 0, e) * factor) * (value(q, 1, e) * factor) * a.alpha;
          }
        };
        if (a.activation == DH_ACT_SILU) {
          gated([](float g) { return act_silu(g); });
          if (a.clamp_max > 0.f)
#pragma unroll
            for (int e = 0; e < 16; e++) v[e] = fminf(fmaxf(v[e], -a.clamp_max), a.clamp_max);
        } else {
          gated([](float g) { return gelu_tanh_fast(g); });
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] = value(q, 0, e) * unscale(row(q, e));
        if (a.ksplit <= 1) {
#pragma unroll
          for (int e = 0; e < 16; e++) v[e] = v[e] * a.alpha + (with_residual ? res[u][e] : 0.f);
        }
      }
      if (n >= a.N) continue;
      auto store = [&](auto* c, auto&& as) {
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int m = m0 + row(q, e);
          if (m < a.M) c[(int64_t)m * a.N + n] = as(v[e]);
        }
      };
      if (!DUAL && a.ksplit > 1) store(a.partial + (int64_t)blockIdx.z * a.M * a.N, [](float x) { return x; });
      else if (a.c_f16) store(reinterpret_cast<__half*>(a.C), [](float x) { return __float2half(x); });
      else store(reinterpret_cast<float*>(a.C), [](float x) { return x; });
    }
  }
}

// T = MFMA tiles per wave along each of M and N (T = 2: a 64 x 64 quadrant per wave, T = 1:
// 32 x 32 when larger tiles would leave most compute units idle).  Four waves cover a
// 64T x 64T tile; MG = groups of four waves stacked along M, all multiplying against the same
// weight tile.  Workgroup tile: 64T MG x 64T.  The weights of a tile are dequantised once per
// workgroup, so MG = 2 halves that work per matrix-core instruction.
template <bool DUAL, int T, int MG>
__global__ __launch_bounds__(256 * MG) void q4k_gemm_kernel(const GemmArgs a) {
  constexpr int NMAT = DUAL ? 2 : 1;
  constexpr int SUBM = 64 * T;                               // rows of one group's A tile
  constexpr int BM = SUBM * MG, BN = 64 * T;
  constexpr int A_HALVES = BM * LDS_ROW, B_HALVES = BN * LDS_ROW;
  extern __shared__ __align__(16) _Float16 lds[];            // [2 buffers][A | B | (B2)]
  constexpr int BUF_HALVES = A_HALVES + NMAT * B_HALVES;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int PT = 256 * MG;                               // threads of the workgroup
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave >> 2) * SUBM + ((wave >> 1) & 1) * 32 * T, wn = (wave & 1) * 32 * T;
  const int fr = lane & 31, fg = lane >> 5;                  // fragment row / k half
  const int64_t row_bytes = (int64_t)a.nb * kBlockBytes;
  const int kt0 = a.ksplit > 1 ? (int)blockIdx.z * a.kt_per_split : 0;
  const int nkt = a.ksplit > 1 ? min((a.K + BK - 1) / BK, kt0 + a.kt_per_split) : (a.K + BK - 1) / BK;

  // ---- global -> register staging
  // A: 16-byte pieces of the packed rows, idx = tid + PT i: row idx >> 3, halves 8 * (idx & 7)
  // W: item (matrix, row, half) = 16 nibble bytes of one row + its block header; SPLIT threads
  //    share an item (QD dwords each) when there are more threads than items
  constexpr int NA = BM * 8 / PT;                            // 16-byte loads of A per thread
  constexpr int ITEMS = 2 * BN * NMAT;
  constexpr int SPLIT = PT > ITEMS ? (PT / ITEMS > 2 ? 2 : PT / ITEMS) : 1;
  constexpr int QD = 4 / SPLIT;                              // dwords of nibbles per thread and item
  constexpr int UNITS = ITEMS * SPLIT;
  constexpr int NW = UNITS > PT ? UNITS / PT : 1;            // units per thread
  constexpr bool ALL_ACTIVE = UNITS >= PT;                   // every producer thread has its units
  static_assert(BM * 8 % PT == 0 && (UNITS % PT == 0 || UNITS < PT), "producer threads must tile the work");
  // per-thread byte offsets of the loads (the host checks that both operands stay below 2 GB)
  uint32_t w_off[NW], a_off[NA];
  bool w_second[NW];
  int w_lds[NW], w_qoff[NW];
  bool w_active[NW];
#pragma unroll
  for (int j = 0; j < NW; j++) {
    const int u = tid + PT * j, it = u / SPLIT, sub = u % SPLIT;
    const int mt = it / (2 * BN), rem = it % (2 * BN), row = rem >> 1, half = rem & 1;
    w_active[j] = u < UNITS;
    w_qoff[j] = 16 + 16 * half + 8 * sub;
    // rows past the tile or the matrix re-read row N - 1: the loads stay unconditional
    // a matrix's units are a multiple of 64 threads: uniform per wave, so the base stays scalar
    w_second[j] = NMAT > 1 && __builtin_amdgcn_readfirstlane(mt & 1) != 0;
    w_off[j] = (uint32_t)((int64_t)min(n0 + row, a.N - 1) * row_bytes);
    w_lds[j] = A_HALVES + (mt % NMAT) * B_HALVES + row * LDS_ROW + 8 * half + 16 * QD * sub;
  }
  // Two register sets: while tile kt is multiplied, tile kt+1 waits in one set and the loads of
  // tile kt+2 are in flight into the other, so a load has two K steps to arrive.
  struct Staged {
    u32x4_t a[NA];
    u32x4_t q[NW], h[NW];
  };
  Staged st0, st1;
  // row factors of this tile's activation rows: one global read each, then LDS
  __shared__ float2 rs_lds[BM];
  for (int r = threadIdx.x; r < BM; r += blockDim.x) rs_lds[r] = a.row_scale[min(m0 + r, a.M - 1)];

  // Every load is unconditional (past the end of K the last tile is loaded again and never used,
  // rows past the matrix re-read its last row): loads complete in order, so with exactly one
  // tile's loads issued per step the wait in front of the older tile leaves the younger tile's
  // loads in flight.  A load under a condition turns that wait into "all loads", and a load then
  // has one K step to arrive instead of two.
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int idx = tid + PT * i, r = idx >> 3;
    a_off[i] = (uint32_t)(((int64_t)min(m0 + r, a.M - 1) * a.kpad + 8 * (idx & 7)) * 2);
  }
  // Buffer loads: address = descriptor base + per-thread 32-bit offset + per-step scalar offset,
  // so the loop holds no vector address arithmetic (and a read past a tensor would return 0).
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16*>(a.Apk), 0, (int)min((int64_t)a.M * a.kpad * 2, (int64_t)0x7fffffff), 0x00020000);
  const int w_bytes = (int)min((int64_t)a.N * row_bytes, (int64_t)0x7fffffff);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W), 0, w_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t w2_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(NMAT > 1 ? a.W2 : a.W), 0, w_bytes, 0x00020000);
  auto load_tile = [&](int kt, Staged& st) {
#pragma unroll
    for (int i = 0; i < NA; i++)
      st.a[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[i], kt * (BK * 2), 0));
    const int blk = kt >> 2, c = kt & 3;
#pragma unroll
    for (int j = 0; j < NW; j++) {
      const __amdgpu_buffer_rsrc_t r = w_second[j] ? w2_rsrc : w_rsrc;
      st.h[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, w_off[j], blk * kBlockBytes, 0));
      if constexpr (QD == 4) {
        st.q[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, w_off[j] + w_qoff[j],
                                                                                  blk * kBlockBytes + 32 * c, 0));
      } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, w_off[j] + w_qoff[j], blk * kBlockBytes + 32 * c, 0);
        st.q[j][0] = v[0];
        st.q[j][1] = v[1];
      }
    }
  };

  float16_t acc[NMAT][T][T];
#pragma unroll
  for (int mt = 0; mt < NMAT; mt++)
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[mt][i][j][e] = 0.f;

  // Multiplies the tile in LDS buffer kt & 1.  Fragments are double-buffered in registers: the
  // reads of k slice ks+1 are issued before the matrix-core instructions of slice ks, so the LDS
  // latency runs under them.  after(slot) is called behind every matrix-core instruction
  // (slot = its index within the K step).
  constexpr int NMFMA = (BK / 16) * NMAT * T * T;
  constexpr int FD = 2;                                      // fragment sets in flight (3 and 4 measured: no gain)
  auto multiply_step = [&](int kt, auto&& after) {
    const _Float16* At = lds + (kt & 1) * BUF_HALVES;
    half8_t af[FD][T], bf[FD][NMAT][T];
    auto read_frags = [&](int ks, half8_t (&fa)[T], half8_t (&fb)[NMAT][T]) {
#pragma unroll
      for (int i = 0; i < T; i++)
        fa[i] = *reinterpret_cast<const half8_t*>(At + (wm + 32 * i + fr) * LDS_ROW + 16 * ks + 8 * fg);
#pragma unroll
      for (int mt = 0; mt < NMAT; mt++)
#pragma unroll
        for (int j = 0; j < T; j++)
          fb[mt][j] = *reinterpret_cast<const half8_t*>(At + A_HALVES + mt * B_HALVES + (wn + 32 * j + fr) * LDS_ROW +
                                                        16 * ks + 8 * fg);
    };
#pragma unroll
    for (int ks = 0; ks < FD - 1; ks++) read_frags(ks, af[ks], bf[ks]);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) {
      if (ks + FD - 1 < BK / 16) read_frags(ks + FD - 1, af[(ks + FD - 1) % FD], bf[(ks + FD - 1) % FD]);
#pragma unroll
      for (int mt = 0; mt < NMAT; mt++)
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
          for (int j = 0; j < T; j++) {
            // accumulators pinned to the accumulation registers: left to itself the compiler keeps
            // them in vector registers and copies all of them aside and back every K step
            asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0"
                         : "+a"(acc[mt][i][j])
                         : "v"(af[ks % FD][i]), "v"(bf[ks % FD][mt][j]));
            after(((ks * NMAT + mt) * T + i) * T + j);
          }
    }
  };
  auto no_hook = [](int) {};

  // The producer's work of one K step in NPARTS pieces, so that it can be dealt out between the
  // matrix-core instructions of the same wave (each runs for 32 cycles while the wave is free to
  // issue vector instructions): piece 0 stores the A tile, then per weight unit the scales and
  // its dwords of nibbles, and the last piece issues the loads two tiles ahead.
  constexpr int NPARTS = 2 + (1 + QD) * NW;
  PairScales ps[NW];
  const Magic magic = magic_numbers();
  auto produce_part = [&](int part, int kt, Staged& nxt) {      // moves tile kt + 1
    _Float16* At = lds + ((kt & 1) ^ 1) * BUF_HALVES;
    if (part == 0) {
#pragma unroll
      for (int i = 0; i < NA; i++) {
        const int idx = tid + PT * i, r = idx >> 3;
        *reinterpret_cast<u32x4_t*>(At + r * LDS_ROW + 8 * (idx & 7)) = nxt.a[i];
      }
    } else if (part == NPARTS - 1) {
      load_tile(min(kt + 3, nkt - 1), nxt);
    } else {
      const int j = (part - 1) / (1 + QD), d = (part - 1) % (1 + QD) - 1;
      if (ALL_ACTIVE || w_active[j]) {
        if (d < 0) {
          ps[j] = pair_scales_f16(nxt.h[j], scale_bits(nxt.h[j], (kt + 1) & 3));
        } else {
          // a dword's eight weights are one piece of the packed k order (packed_place)
          uint4 w;
          dequant_low(nxt.q[j][d], ps[j], magic, w.x, w.y);
          dequant_high(nxt.q[j][d], ps[j], magic, w.z, w.w);
          *reinterpret_cast<uint4*>(At + w_lds[j] + 16 * d) = w;
        }
      }
    }
  };
  auto produce_first = [&]() {
    load_tile(kt0, st0);
#pragma unroll
    for (int part = 0; part < NPARTS - 1; part++) produce_part(part, kt0 - 1, st0);   // tile kt0 into its buffer
    load_tile(min(kt0 + 1, nkt - 1), st0);
    load_tile(min(kt0 + 2, nkt - 1), st1);
  };
  // Multiplies tile kt and, between its matrix-core instructions, moves tile kt+1 out of `nxt`
  // into the other LDS buffer and reloads `nxt` with tile kt+3.
  auto fused_step = [&](int kt, Staged& nxt) {
    multiply_step(kt, [&](int slot) {
#pragma unroll
      for (int part = 0; part < NPARTS; part++)
        if (part * NMFMA / NPARTS == slot) produce_part(part, kt, nxt);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  produce_first();
  __syncthreads();
  int kt = kt0;
  for (; kt + 2 < nkt; kt += 2) {        // st0 holds the tiles at odd distance from kt0, st1 the even ones
    fused_step(kt, st0);
    __syncthreads();
    fused_step(kt + 1, st1);
    __syncthreads();
  }
  if (kt + 1 < nkt) {
    fused_step(kt, st0);
    __syncthreads();
    kt++;
  }
  multiply_step(kt, no_hook);

  // the matrix-core instructions above are inline asm, invisible to the compiler's hazard
  // checks: give the last one time to retire before its accumulators are read
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  store_results<DUAL, T * T>(
      a, m0, [&](int q, int matrix, int e) { return acc[DUAL ? matrix : 0][q / T][q % T][e]; },
      [&](int q, int e) { return wm + 32 * (q / T) + 8 * (e >> 2) + 4 * fg + (e & 3); }, [&](int q) { return n0 + wn + 32 * (q % T) + fr; },
      [&](int row) { return rs_lds[row].y; });
}

// ---- the wide kernel
// WM x WN waves; a wave computes 32 RA rows x 64 columns (DUAL: 32 columns of both matrices).  KG such groups of waves, each with tiles of its own,
// take runs of the super-blocks; their sums meet in LDS at the end.
template <int WM_, int WN_, int RA_>
struct Q4Tile {
  static constexpr int WM = WM_, WN = WN_, RA = RA_;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int BM = 32 * RA * WM, kRows = 64 * WN;                // weight rows of a tile (of both matrices together)
  static constexpr int kBufA = BM * 128, kRoundsA = kBufA / (1024 * kWaves);
  static constexpr int kRowsWave = kRows / kWaves;                        // weight rows a wave fetches: 144 bytes each
  static constexpr int kRoundsB = (kRowsWave * 9 + 63) / 64, kRegion = kRoundsB * 1024, kBufB = kRegion * kWaves;
  static constexpr int kLds = 2 * (kBufA + kBufB);
  static_assert(kBufA % (1024 * kWaves) == 0 && kRowsWave <= 32 * WN && kRowsWave % 32 == 0, "whole loads; a wave fetches rows of one matrix");
};

template <class Tile, bool DUAL, int KG>
__global__ __launch_bounds__(Tile::kThreads * KG, 2) void q4k_wide_kernel(const GemmArgs a) {
  constexpr int RA = Tile::RA, WN = Tile::WN, NB = Tile::kRoundsB, NA = Tile::kRoundsA;
  constexpr int BN = DUAL ? Tile::kRows / 2 : Tile::kRows;
  extern __shared__ __align__(16) char smem_all[];
  __shared__ float rs_lds[Tile::BM];
  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = KG > 1 ? wave_all / Tile::kWaves : 0, wave = wave_all - group * Tile::kWaves;
  char* const smem = smem_all + group * Tile::kLds;
  const int wm = wave / WN, wn = wave % WN;
  const int tile = dh::xcd_contiguous(blockIdx.x, a.tiles_m * a.tiles_n);
  const int m0 = (tile % a.tiles_m) * Tile::BM, n0 = (tile / a.tiles_m) * BN;
  const int fr = lane & 31, fh = lane >> 5;
  const int kt_first = a.ksplit > 1 ? (int)blockIdx.z * a.kt_per_split : 0;    // a multiple of 4
  const int steps = (a.ksplit > 1 ? min((a.K + BK - 1) / BK, kt_first + a.kt_per_split) : (a.K + BK - 1) / BK) - kt_first;
  // a group's steps: whole super-blocks, at least one (the host sees to KG of them)
  auto group_first = [&](int g) { return min((steps + 3) / 4 * g / KG * 4, steps); };
  const int kt0 = kt_first + group_first(group), nk = group_first(group + 1) - group_first(group);
  const int sb0 = kt0 >> 2, sb_last = (kt0 + nk - 1) >> 2;
  for (int r = threadIdx.x; r < Tile::BM; r += Tile::kThreads * KG) rs_lds[r] = a.row_scale[min(m0 + r, a.M - 1)].y;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // ---- fetches
  uint32_t va[NA], vb[NB];
  {
    const int row_lane = 8 * wave + (lane >> 3);
    const uint32_t piece = 16 * ((lane & 7) ^ ((row_lane >> 1) & 7));
#pragma unroll
    for (int r = 0; r < NA; r++) {
      const int row = 8 * Tile::kWaves * r + row_lane;
      va[r] = (uint32_t)min(row, a.M - 1 - m0) * (uint32_t)a.kpad * 2u + piece;
    }
  }
  const int row_first = wave * Tile::kRowsWave;                            // among the tile's: matrix (or column group) first
  const int frag_first = row_first / (32 * WN);
  const int64_t row_bytes = (int64_t)a.nb * kBlockBytes;
#pragma unroll
  for (int r = 0; r < NB; r++) {
    const int at = min(64 * r + lane, Tile::kRowsWave * 9 - 1);            // past the rows: the last piece again
    const int row = row_first % (32 * WN) + at / 9;                        // column group row / 32 of this fragment, column row % 32
    const int n = DUAL ? row : (row >> 5) * 64 + 32 * frag_first + (row & 31);
    vb[r] = (uint32_t)((int64_t)min(n, a.N - 1 - n0) * row_bytes) + 16u * (at % 9);
  }
  const dh::buffer_words_t wa = dh::buffer_words(a.Apk + (int64_t)m0 * a.kpad);
  const dh::buffer_words_t wb = dh::buffer_words((DUAL && frag_first ? a.W2 : a.W) + (int64_t)n0 * row_bytes);
  const uint32_t lds_a = lds0 + 1024 * wave, lds_b = lds0 + 2 * Tile::kBufA + Tile::kRegion * wave;
  auto fetch_a = [&](int t, int buf) {
    const uint32_t k = 128u * (uint32_t)(kt0 + min(t, nk - 1));
#pragma unroll
    for (int r = 0; r < NA; r++) dh::fetch_to_lds(wa, va[r], k, lds_a + buf * Tile::kBufA + 1024 * Tile::kWaves * r);
  };
  auto fetch_b = [&](int r, uint32_t k, uint32_t buf_at) { dh::fetch_to_lds(wb, vb[r], k, lds_b + buf_at + 1024 * r); };
  auto b_at = [&](int sb) { return (uint32_t)min(sb, sb_last) * kBlockBytes; };

  // ---- LDS reads
  const char* ra[4];
#pragma unroll
  for (int ks = 0; ks < 4; ks++) ra[ks] = smem + (32 * RA * wm + fr) * 128 + 16 * ((2 * ks + fh) ^ ((fr >> 1) & 7));
  const char* rb[2];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const int row = f * 32 * WN + 32 * wn + fr;
    rb[f] = smem + 2 * Tile::kBufA + row / Tile::kRowsWave * Tile::kRegion + row % Tile::kRowsWave * kBlockBytes;
  }
  u32x4_t fa[2][RA], raw[2][2], hdr[2], fb[2][2];
  PairScales ps[2][2];
  ScaleBits bits;
  const Magic magic = magic_numbers();
  float16_t acc[RA][2];
#pragma unroll
  for (int i = 0; i < RA; i++)
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][f][e] = 0.f;

  auto read_a = [&](int buf, int ks, int set) {
#pragma unroll
    for (int i = 0; i < RA; i++) fa[set][i] = *reinterpret_cast<const u32x4_t*>(ra[ks] + buf * Tile::kBufA + i * 4096);
  };
  auto read_b = [&](int c, uint32_t buf_at, int set) {
#pragma unroll
    for (int f = 0; f < 2; f++) {
      hdr[f] = *reinterpret_cast<const u32x4_t*>(rb[f] + buf_at);
      raw[set][f] = *reinterpret_cast<const u32x4_t*>(rb[f] + buf_at + 16 + 32 * c + 16 * fh);
    }
  };
  // A slice's weights of fragment f in three stages of independent instructions (a dependent one waits eight cycles for its operand, so
  // four chains side by side, with matrix-core instructions between the stages, take half the time of one after the other): the nibbles
  // under their exponents, the numbers themselves, the weights.
  half2_t nib[2][4];
  auto dequant = [&](int stage, int f, int ks, int step_set, int set) {
    const half2_t k1024 = {(_Float16)1024.f, (_Float16)1024.f}, k64 = {(_Float16)64.f, (_Float16)64.f};
    half2_t(&v)[4] = nib[f];
    const PairScales& p = ps[step_set][f];
    if (stage == 0) {
      const uint32_t w = raw[step_set][f][ks], w8 = w >> 8;
      v[0] = __builtin_bit_cast(half2_t, (w & 0x000F000Fu) | magic.low);
      v[2] = __builtin_bit_cast(half2_t, (w & 0x00F000F0u) | magic.high);
      v[1] = __builtin_bit_cast(half2_t, (w8 & 0x000F000Fu) | magic.low);
      v[3] = __builtin_bit_cast(half2_t, (w8 & 0x00F000F0u) | magic.high);
    } else if (stage == 1) {
      v[0] = v[0] - k1024; v[2] = v[2] - k64; v[1] = v[1] - k1024; v[3] = v[3] - k64;
    } else {
      fb[set][f][0] = __builtin_bit_cast(uint32_t, v[0] * p.slo + p.mlo);
      fb[set][f][2] = __builtin_bit_cast(uint32_t, v[2] * p.shi + p.mhi);
      fb[set][f][1] = __builtin_bit_cast(uint32_t, v[1] * p.slo + p.mlo);
      fb[set][f][3] = __builtin_bit_cast(uint32_t, v[3] * p.shi + p.mhi);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int NM = 2 * RA;
  // multiplies slice ks; behind its matrix-core instruction n `between(n)` is called
  auto multiply = [&](int ks, auto&& between) {
    int n = 0;
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int i = 0; i < RA; i++) {
        acc[i][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, fa[ks & 1][i]), __builtin_bit_cast(half8_t, fb[ks & 1][f]),
                                                           acc[i][f], 0, 0, 0);
        between(n++);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  // b_now, b_next: where this super-block and the next lie in LDS; k_next: the next one's place in its row
  auto step = [&](int t, auto chunk, uint32_t b_now, uint32_t b_next, uint32_t k_next) {
    constexpr int C = decltype(chunk)::value, P = C & 1, Q = P ^ 1;
    constexpr int per = (NB + 1) / 2, lo = C == 0 ? 0 : C == 1 ? per : NB, hi = C == 0 ? per : NB;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      if (ks == 3) dh::arrive_and_wait<hi - lo>();     // step t + 1's activations are there, and with step 2's all of the next super-block
      multiply(ks, [&](int n) {
        if (n == 0) {
          if (ks < 3) {
            read_a(P, ks + 1, (ks + 1) & 1);
          } else {
            read_a(Q, 0, 0);
            fetch_a(t + 2, P);
          }
          if (ks == 0) read_b((C + 1) & 3, C == 3 ? b_next : b_now, Q);
        }
        if (ks < 3)
          for (int r = lo + ks; r < hi; r += 3)
            if (n == (r - lo) / 3) fetch_b(r, k_next, b_next);
        // the next slice's weights; in the middle two slices the next step's scales
        const int next_ks = (ks + 1) & 3, src = ks < 3 ? P : Q, dst = (ks + 1) & 1;
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
          for (int stage = 0; stage < 3; stage++)
            if (n == (NM == 2 ? stage / 2 : NM == 4 ? f + stage : 3 * f + stage)) dequant(stage, f, next_ks, src, dst);
        if (ks == 1 || ks == 2) {
          if (n == (NM <= 4 ? 0 : 6)) bits = scale_bits(hdr[ks - 1], (C + 1) & 3);
          if (n == NM - 1) ps[Q][ks - 1] = pair_scales_f16(hdr[ks - 1], bits);
        }
      });
    }
  };

#pragma unroll
  for (int r = 0; r < NB; r++) fetch_b(r, b_at(sb0), 0);
  fetch_a(0, 0);
  fetch_a(1, 1);
  dh::arrive_and_wait<NA>();
  read_b(0, 0, 0);
  read_a(0, 0, 0);
#pragma unroll
  for (int f = 0; f < 2; f++) ps[0][f] = pair_scales_f16(hdr[f], scale_bits(hdr[f], 0));
#pragma unroll
  for (int f = 0; f < 2; f++)
#pragma unroll
    for (int stage = 0; stage < 3; stage++) dequant(stage, f, 0, 0, 0);
  uint32_t now = 0, next = Tile::kBufB;
  for (int t = 0, sb = sb0;; t += 4, sb++) {
    const uint32_t k_next = b_at(sb + 1);
    step(t, std::integral_constant<int, 0>{}, now, next, k_next);
    if (t + 1 >= nk) break;
    step(t + 1, std::integral_constant<int, 1>{}, now, next, k_next);
    if (t + 2 >= nk) break;
    step(t + 2, std::integral_constant<int, 2>{}, now, next, k_next);
    if (t + 3 >= nk) break;
    step(t + 3, std::integral_constant<int, 3>{}, now, next, k_next);
    if (t + 4 >= nk) break;
    const uint32_t was = now;
    now = next;
    next = was;
  }
  if constexpr (KG > 1) {                  // steps that other groups have more
    int most = 0;
#pragma unroll
    for (int g = 0; g < KG; g++) most = max(most, group_first(g + 1) - group_first(g));
    for (int i = nk; i < most; i++) dh::arrive_and_wait<0>();
  }
  dh::arrive_and_wait<0>();                // nothing may be in flight towards LDS when the workgroup ends
  if constexpr (KG > 1) {
    // the other groups' sums go where their tiles were and are added in group order
    static_assert(RA * 2 * 64 * Tile::kThreads <= Tile::kLds, "a group's sums fit where its tiles were");
    auto sums_of = [&](int g) { return reinterpret_cast<float4*>(smem_all + g * Tile::kLds) + (wave * 64 + lane); };
    if (group > 0) {
#pragma unroll
      for (int q = 0; q < 2 * RA; q++)
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
          const float16_t& v = acc[q >> 1][q & 1];
          sums_of(group)[(4 * q + e / 4) * Tile::kThreads] = make_float4(v[e], v[e + 1], v[e + 2], v[e + 3]);
        }
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KG; g++)
#pragma unroll
      for (int q = 0; q < 2 * RA; q++)
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
          float16_t& v = acc[q >> 1][q & 1];
          const float4 other = sums_of(g)[(4 * q + e / 4) * Tile::kThreads];
          v[e] += other.x; v[e + 1] += other.y; v[e + 2] += other.z; v[e + 3] += other.w;
        }
  }

  store_results<DUAL, DUAL ? RA : 2 * RA>(
      a, m0, [&](int q, int matrix, int e) { return DUAL ? acc[q][matrix][e] : acc[q >> 1][q & 1][e]; },
      [&](int q, int e) { return 32 * (RA * wm + (DUAL ? q : q >> 1)) + 4 * fh + 8 * (e >> 2) + (e & 3); },
      [&](int q) { return n0 + (DUAL ? 32 * wn : 64 * wn + 32 * (q & 1)) + fr; }, [&](int row) { return rs_lds[row]; });
}

// C = alpha * (sum of the split-K pieces, in split order) + residual.  Four consecutive outputs per
// thread when the row length allows 16-byte accesses, every piece's load in flight before the sums.
constexpr int kMaxSplit = 8;
template <bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const GemmArgs a) {
  const int64_t total = (int64_t)a.M * a.N;
  constexpr int W = VEC ? 4 : 1;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * W;
  if (i >= total) return;
  float p[kMaxSplit][W];
#pragma unroll
  for (int z = 0; z < kMaxSplit; z++) {
    if (z < a.ksplit) {
      if constexpr (VEC) {
        const float4 t = *reinterpret_cast<const float4*>(a.partial + (int64_t)z * total + i);
        p[z][0] = t.x; p[z][1] = t.y; p[z][2] = t.z; p[z][3] = t.w;
      } else {
        p[z][0] = a.partial[(int64_t)z * total + i];
      }
    }
  }
  float r[W];
#pragma unroll
  for (int e = 0; e < W; e++) r[e] = 0.f;
  if (a.residual) {
    if constexpr (VEC) {
      const float4 t = *reinterpret_cast<const float4*>(a.residual + i);
      r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else {
      r[0] = a.residual[i];
    }
  }
#pragma unroll
  for (int e = 0; e < W; e++) {
    float s = 0.f;
#pragma unroll
    for (int z = 0; z < kMaxSplit; z++)
      if (z < a.ksplit) s += p[z][e];
    r[e] = s * a.alpha + r[e];
  }
  if (a.c_f16) {
    __half* c = reinterpret_cast<__half*>(a.C) + i;
#pragma unroll
    for (int e = 0; e < W; e++) c[e] = __float2half(r[e]);
  } else if constexpr (VEC) {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.C) + i) = make_float4(r[0], r[1], r[2], r[3]);
  } else {
    reinterpret_cast<float*>(a.C)[i] = r[0];
  }
}

int launch_reduce(const GemmArgs& a, const char* op) {
  const int64_t total = (int64_t)a.M * a.N;
  if (a.ksplit > kMaxSplit) return dh::fail(2, "[%s] internal: K cut into %d pieces, the reduction takes %d", op, a.ksplit, kMaxSplit);
  const bool vec = total % 4 == 0 && (reinterpret_cast<uintptr_t>(a.C) | reinterpret_cast<uintptr_t>(a.residual)) % 16 == 0;
  if (vec)
    hipLaunchKernelGGL(splitk_reduce_kernel<true>, dim3((unsigned)dh::ceil_div(total / 4, 256)), dim3(256), 0, dh::stream(), a);
  else
    hipLaunchKernelGGL(splitk_reduce_kernel<false>, dim3((unsigned)dh::ceil_div(total, 256)), dim3(256), 0, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

template <bool DUAL, int T, int MG>
int launch_gemm_cfg(const GemmArgs& a, const char* op) {
  constexpr int BM = 64 * T * MG, BN = 64 * T;
  const size_t lds = (size_t)2 * (BM + (DUAL ? 2 : 1) * BN) * LDS_ROW * sizeof(_Float16);
  auto kern = q4k_gemm_kernel<DUAL, T, MG>;
  static bool attr_set = false;   // once per instantiation: the call costs microseconds
  if (!attr_set) {
    DH_CHECK_HIP(op, hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set = true;
  }
  const dim3 grid((unsigned)dh::ceil_div(a.N, BN), (unsigned)dh::ceil_div(a.M, BM), (unsigned)std::max(1, a.ksplit));
  hipLaunchKernelGGL(kern, grid, dim3(256 * MG), lds, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return a.ksplit > 1 ? launch_reduce(a, op) : 0;
}

template <class Tile, bool DUAL, int KG = 1>
int launch_wide(GemmArgs a, const char* op) {
  auto kern = q4k_wide_kernel<Tile, DUAL, KG>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, KG * Tile::kLds);
  DH_CHECK_HIP(op, set);
  a.tiles_m = (int)dh::ceil_div(a.M, Tile::BM);
  a.tiles_n = (int)dh::ceil_div(a.N, DUAL ? Tile::kRows / 2 : Tile::kRows);
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.tiles_m * a.tiles_n), 1, (unsigned)std::max(1, a.ksplit)), dim3(Tile::kThreads * KG), KG * Tile::kLds, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

// Tiles of q4k_wide_kernel and what 64 k of one cost in ns, with few workgroups on the device, with one on every compute unit, with as many
// as fit; start: outside the k loop.  Fitted to M = 64 .. 2048 over the products of models 1024 .. 4096 wide.
struct WideCost {
  int bm, rows, per_cu;
  float alone, one, full, start;
};
constexpr WideCost kWide[] = {{256, 256, 1, 1200.f, 1950.f, 1950.f, 8000.f},       // <2, 4, 4>
                              {128, 256, 1, 760.f, 1120.f, 1250.f, 9000.f},        // <1, 4, 4>
                              {128, 256, 1, 845.f, 1200.f, 1250.f, 5500.f},        // <2, 4, 2>
                              {128, 128, 2, 580.f, 720.f, 1280.f, 5000.f}};        // <2, 2, 2>
struct WideChoice {
  int tile, pieces;
};
// The cheapest of them, with K cut in pieces (of whole super-blocks) where that pays for the reduction.
WideChoice choose_wide(int64_t M, int64_t N, int64_t K, bool dual) {
  const int64_t cus = dh::num_cus(), steps = dh::ceil_div(K, BK);
  size_t ws_bytes = 0;
  (void)dh::splitk_workspace(&ws_bytes);
  const int most = dual ? 1 : (int)std::max<size_t>(1, std::min<size_t>(kMaxSplit, ws_bytes / ((size_t)M * N * sizeof(float))));
  WideChoice best{0, 1};
  double least = 1e30;
  for (int i = 0; i < 4; i++) {
    const WideCost& c = kWide[i];
    for (int s = 1; s <= most && (s == 1 || steps >= 8 * s); s++) {
      const int64_t groups = dh::ceil_div(M, c.bm) * dh::ceil_div(N, dual ? c.rows / 2 : c.rows) * s, slots = cus * c.per_cu, left = groups % slots;
      const double f = (double)left / cus;
      const double step = f <= 1.0 ? c.alone + (c.one - c.alone) * f : c.full * (0.85 + 0.15 * f / c.per_cu);
      double t = 4.0 * dh::ceil_div(steps, 4 * s) * ((double)(groups / slots) * c.full + (left ? step : 0.0)) + c.start;
      if (s > 1) t += 3500.0 + 4.0 * M * N * (2 * s + 1) / 4000.0;
      if (t < least) {
        least = t;
        best = WideChoice{i, s};
      }
    }
  }
  const int env_tile = dh::tuning_int("DH_Q4_TILE", -1);
  if (env_tile >= 0) best.tile = env_tile;
  return best;
}
// Steps of 64 k in a piece.
int64_t steps_per_piece(int64_t K, int pieces) { return dh::ceil_div(dh::ceil_div(K, BK), 4 * pieces) * 4; }

void cut(GemmArgs& a, int pieces) {
  if (pieces <= 1) return;
  a.kt_per_split = (int)steps_per_piece(a.K, pieces);
  a.ksplit = (int)dh::ceil_div(dh::ceil_div(a.K, BK), a.kt_per_split);
  size_t ws_bytes = 0;
  if (a.ksplit > 1) a.partial = dh::splitk_workspace(&ws_bytes);
}

template <bool DUAL>
int launch_wide_best(GemmArgs a, const char* op) {
  const WideChoice pick = choose_wide(a.M, a.N, a.K, DUAL);
  cut(a, pick.pieces);
  int rc;
  switch (pick.tile) {
    case 0: rc = launch_wide<Q4Tile<2, 4, 4>, DUAL>(a, op); break;
    case 1: rc = launch_wide<Q4Tile<1, 4, 4>, DUAL>(a, op); break;
    case 2: rc = launch_wide<Q4Tile<2, 4, 2>, DUAL>(a, op); break;
    default: rc = launch_wide<Q4Tile<2, 2, 2>, DUAL>(a, op); break;
  }
  return rc || a.ksplit <= 1 ? rc : launch_reduce(a, op);
}

// Products of enough work, or of enough tiles, go to q4k_wide_kernel's large tiles: where a step's latency counts instead of its throughput the other
// kernel is ahead, because its waves share one dequantised tile (us, that one / the wide one, weights from memory: 128 x 1152 x 6912 20 / 28,
// 512 x 1152 x 6912 33.2 / 33.2, but 1024 x 2048 x 1024 25.3 / 24.3, 200 x 6144 x 4096 39.5 / 37.3, 512 x 4096 x 12288
// 142 / 82; a threshold of the product's size, as the costs of the other kernel are not in the table: over 236 shapes 1.5 % behind the best).  Pairs of
// few steps stay there at any height (2048 x 1024 x 512 18 / 21, 1024 x 2048 x 1024 22 / 24).
bool takes_wide(int64_t M, int64_t N, int64_t K, bool dual) {
  return dh::ceil_div(M, 256) * dh::ceil_div(N, 128) >= dh::num_cus() || (double)M * N * K * (dual ? 2 : 1) >= (M >= 1024 && !dual ? 2e9 : 5e9);
}

// Pieces of K with which 128 x 128 tiles of q4k_gemm_kernel occupy half of the compute units, or 0 where no number of them does.
int big_tile_pieces(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = dh::num_cus(), tiles = dh::ceil_div(M, 128) * dh::ceil_div(N, 128);
  if (2 * tiles >= cus) return 1;
  size_t ws_bytes = 0;
  (void)dh::splitk_workspace(&ws_bytes);
  int64_t pieces = std::min<int64_t>({8, cus / tiles, dh::ceil_div(K, BK) / 8});
  while (pieces > 1 && (size_t)pieces * M * N * sizeof(float) > ws_bytes) pieces--;
  return pieces > 1 && 2 * tiles * pieces >= cus ? (int)pieces : 0;
}

// Few rows: q4k_wide_kernel on tiles of 32 or 64 rows x 128 weight rows (two waves), two such groups along k (three: 35.3 -> 37.8 us for the
// pair of 64 x 12288 x 4096, their waves do not divide among four SIMDs).  There a weight is dequantised once, in the registers of the wave that
// multiplies it, and read from LDS as nibbles; q4k_gemm_kernel writes and reads it there as f16 and reads the activations for every 32 columns: 72 KB a
// step of 64 k, which at 128 bytes a clock is most of its 0.6 us, whatever the number of rows.  us with packing and reduction, weights from memory, before
// / now: pairs 16 x 12288 x 4096 42.6 / 30.3, 64 x 12288 x 4096 44 / 35, 40 x 6144 x 2048 24.3 / 18.0, 33 x 3072 x 1024 14.5 / 12.0, 512 x 1024 x 4096 40.8 / 30.3;
// products 16 x 4096 x 4096 17.6 / 14.5, 20 x 4096 x 12288 29.2 / 21.6, 64 x 12288 x 2048 25.0 / 18.2, 16 x 28672 x 4096 51 / 30.
// What a super-block costs a group was fitted to those (3.0 us on 32 rows, 3.7 on 64), as long as the tiles run at once, or on 32 rows in two rounds of more than
// a short k (23 x 35392 x 296 13.5 / 15.4, 18 x 38689 x 532 17.6 / 18.3, 28 x 51643 x 788 23.6 / 23.2, 32 x 60197 x 1088 30.2 / 26.4; pairs 23 x 24571 x 312 13.4 /
// 13.9, 25 x 25711 x 348 14.6 / 14.2, 16 x 21498 x 1520 33.3 / 25.1).  Where the lines lie: pairs of
// over 512 rows (796 x 1536 x 1472 27.7 / 28.2) or under 1024 k on 64-row tiles (170 x 5000 x 640 13.3 / 14.1), products of under 8e6 weights or 2048 columns (64 x 2048 x 2048 12.0 / 13.2, 16 x 2048 x 3072 11.8 / 12.3,
// but 16 x 2048 x 4096 16.1 / 12.6; 54 x 1536 x 5504 15.3 / 16.4), where the other kernel has 64 x 64 tiles, whose pieces of K overlap one another's waits (20 x
// 2609 x 3172 12.6 / 16.0, 59 x 3612 x 2388 14.1 / 16.4, 32 x 16227 x 716 10.8 / 11.7, and with its 128-row tiles 26 x 3998 x 2228 16.8 / 14.3; of over 64 rows it
// has two of them, 70 x 16044 x 612 12.0 / 13.5, 122 x 3957 x 2480 18.3 / 19.6, but from 1024 to 2047 k 94 x 7832 x 1040 16.0 / 12.4, 119 x 4521 x 1872 17.7 / 15.9), of
// over 64 rows that take long (122 x 8448 x 8448 42 / 54, 67 x 6208 x 8320 32.6 / 36.9, but
// 100 x 12000 x 2000 27.1 / 21.0, 128 x 2048 x 6144 25.3 / 21.3).
constexpr int kNarrowGroups = 2;
struct NarrowChoice {
  int bm, pieces;                // rows of a tile (0: another kernel serves the product), pieces of K
};
NarrowChoice choose_narrow(int64_t M, int64_t N, int64_t K, bool dual) {
  const int64_t cus = dh::num_cus(), blocks = dh::ceil_div(K, kQK);
  if (blocks < kNarrowGroups) return {0, 1};
  if (dual ? M > 512 : M > 128 || N < 2048 || N * K < 8000000) return {0, 1};
  if (!dual && K >= 512 && !(M > 64 && K >= 1024 && K < 2048) && big_tile_pieces(M, N, K) == 0) return {0, 1};
  size_t ws_bytes = 0;
  (void)dh::splitk_workspace(&ws_bytes);
  const int64_t most = dual ? 1 : std::min<int64_t>({kMaxSplit, blocks / kNarrowGroups, std::max<int64_t>(1, ws_bytes / ((size_t)M * N * sizeof(float)))});
  NarrowChoice best{0, 1};
  double least = !dual && M > 64 ? 20000.0 : 1e30;
  for (int bm = 32; bm <= 64; bm += 32) {
    const int64_t groups = dh::ceil_div(M, bm) * dh::ceil_div(N, dual ? 64 : 128);
    if (dual && bm == 64 && K < 1024) break;
    for (int64_t s = 1; s <= most; s++) {
      const int64_t each = steps_per_piece(K, (int)s) / 4, pieces = dh::ceil_div(blocks, each), rounds = dh::ceil_div(groups * pieces, cus);
      if (rounds > (M <= 32 && s == 1 && K >= (dual ? 340 : 768) ? 2 : 1)) break;
      if (blocks - each * (pieces - 1) < kNarrowGroups) continue;         // the last piece, too, has a super-block for each group
      double t = (double)rounds * dh::ceil_div(each, kNarrowGroups) * (bm == 32 ? 3000.0 : 3700.0);
      if (pieces > 1) t += 3500.0 + 4.0 * M * N * (2 * pieces + 1) / 4000.0;
      if (t < least) {
        least = t;
        best = NarrowChoice{bm, (int)s};
      }
    }
  }
  return best;
}

// 128 x 128 tiles when they occupy at least half of the compute units (their higher matrix-core
// share wins from there on), else 64 x 64.
template <bool DUAL>
int launch_gemm(GemmArgs a, const char* op) {
  // rows beyond the capacity of the packed-activation scratch go in further passes
  a.kpad = (a.K + BK - 1) / BK * BK;
  if (a.norm_weight && a.K > 16384)
    return dh::fail(1, "[%s] the RMSNorm prologue serves K <= 16384 at M >= 16 (K=%d)", op, a.K);
  // the kernel addresses a weight row as a 32-bit byte offset into a buffer descriptor
  if ((int64_t)a.N * a.nb * kBlockBytes >= ((int64_t)1 << 31))
    return dh::fail(1, "[%s] a weight tensor of %d x %d (2 GB or more) is beyond the prefill GEMM; split it by rows", op,
                    a.N, a.K);
  if (dh::plan_note(DH_PLAN_GEMM)) return 0;
  size_t pk_bytes = 0;
  _Float16* packed = reinterpret_cast<_Float16*>(dh::gemm_packed_a(&pk_bytes));
  float2* scales = reinterpret_cast<float2*>(dh::gemm_row_scale());
  if (!packed || !scales) return dh::fail(2, "[%s] the library's scratch buffers are missing (dh_init)", op);
  const int cap = (int)std::min<size_t>((size_t)dh::gemm_row_scale_capacity(), pk_bytes / ((size_t)a.kpad * 2));
  if (cap < 16) return dh::fail(1, "[%s] K=%d is too long for the prefill GEMM's activation scratch", op, a.K);
  if (a.M > cap) {
    const size_t c_elem = a.c_f16 ? 2 : 4;
    for (int m0 = 0; m0 < a.M; m0 += cap) {
      GemmArgs b = a;
      b.M = std::min(cap, a.M - m0);
      b.A = a.A + (int64_t)m0 * a.K;
      b.C = static_cast<char*>(a.C) + (int64_t)m0 * a.N * c_elem;
      b.residual = a.residual ? a.residual + (int64_t)m0 * a.N : nullptr;
      const int rc = launch_gemm<DUAL>(b, op);
      if (rc) return rc;
    }
    return 0;
  }
#define DH_PACK_ROWS(NV_, THREADS_)                                                                          \
  hipLaunchKernelGGL((pack_a_row_kernel<NV_, THREADS_>), dim3((unsigned)a.M), dim3(THREADS_), 0, dh::stream(), a.A, a.M, a.K, \
                     a.kpad, packed, scales, a.norm_weight, a.norm_eps, a.norm_weight_offset)
  if (a.K <= 2048) DH_PACK_ROWS(2, 256);
  else if (a.K <= 4096) DH_PACK_ROWS(4, 256);
  else if (a.K <= 8192) DH_PACK_ROWS(8, 256);
  else if (a.K <= 16384) DH_PACK_ROWS(4, 1024);
  else if (a.norm_weight)
    return dh::fail(1, "[%s] the RMSNorm prologue serves K <= 16384 at M >= 16 (K=%d)", op, a.K);
  else
    hipLaunchKernelGGL(pack_a_kernel, dim3((unsigned)dh::ceil_div(a.M, 4)), dim3(256), 0, dh::stream(), a.A, a.M, a.K,
                       a.kpad, packed, scales);
#undef DH_PACK_ROWS
  DH_CHECK_LAUNCH(op);
  a.row_scale = scales;
  a.Apk = packed;
  a.ksplit = 1;
  if (const NarrowChoice pick = choose_narrow(a.M, a.N, a.K, DUAL); pick.bm > 0) {
    cut(a, pick.pieces);
    const int rc = pick.bm == 32 ? launch_wide<Q4Tile<1, 2, 1>, DUAL, kNarrowGroups>(a, op) : launch_wide<Q4Tile<1, 2, 2>, DUAL, kNarrowGroups>(a, op);
    return rc || a.ksplit <= 1 ? rc : launch_reduce(a, op);
  }
  if (takes_wide(a.M, a.N, a.K, DUAL)) return launch_wide_best<DUAL>(a, op);
  // The other kernel: for the fused gate/up pair 128 x 64 tiles (eight waves), then 128 x 128 (four waves, two workgroups per compute
  // unit) when those occupy at least half of the compute units, else 64 x 64.
  const int64_t big_tiles = dh::ceil_div(a.M, 128) * dh::ceil_div(a.N, 128);
  if (2 * big_tiles >= dh::num_cus()) {
    if constexpr (DUAL) {
      return launch_gemm_cfg<true, 1, 2>(a, op);
    } else {
      return launch_gemm_cfg<false, 2, 1>(a, op);
    }
  }
  // Few tiles and a long K: every workgroup would walk K alone at one memory round trip per
  // step.  Cut K so that about three workgroups share a compute unit and overlap each other's
  // waits; the pieces meet in the library's scratch buffer.
  if (!DUAL) {
    static const int env_split = env_ksplit();
    static const int env_big = dh::tuning_int("DH_GEMM_BIGSPLIT", 1);
    // 128 x 128 tiles with K cut into pieces when that fills the compute units: their matrix-core
    // share is higher than that of 64 x 64 tiles
    if (env_big) {
      const int nkt = (a.K + BK - 1) / BK, split = big_tile_pieces(a.M, a.N, a.K);
      size_t ws_bytes = 0;
      float* ws = dh::splitk_workspace(&ws_bytes);
      if (split > 1 && ws) {
        a.kt_per_split = (int)dh::ceil_div(nkt, split);
        a.ksplit = (int)dh::ceil_div(nkt, a.kt_per_split);
        a.partial = ws;
        return launch_gemm_cfg<false, 2, 1>(a, op);
      }
    }
    const int64_t tiles = dh::ceil_div(a.M, 64) * dh::ceil_div(a.N, 64);
    const int nkt = (a.K + BK - 1) / BK;
    size_t ws_bytes = 0;
    float* ws = dh::splitk_workspace(&ws_bytes);
    int split = (int)std::min<int64_t>(8, dh::ceil_div(3 * (int64_t)dh::num_cus(), tiles));
    split = std::min(split, nkt / 8);
    if (env_split > 0) split = env_split;
    while (split > 1 && (size_t)split * a.M * a.N * sizeof(float) > ws_bytes) split--;
    if (split > 1 && ws) {
      a.kt_per_split = (int)dh::ceil_div(nkt, split);
      a.ksplit = (int)dh::ceil_div(nkt, a.kt_per_split);
      a.partial = ws;
    }
  }
  return launch_gemm_cfg<DUAL, 1, 1>(a, op);
}

}  // namespace


namespace dh {

int q4k_sum_slices(const char* op, float* parts, int slices, void* C, int c_f16, int M, int N, float alpha, const float* residual) {
  GemmArgs a{};
  a.partial = parts; a.ksplit = slices; a.C = C; a.c_f16 = c_f16; a.M = M; a.N = N; a.alpha = alpha; a.residual = residual;
  return launch_reduce(a, op);
}

bool q4k_gemm_serves(int M, int K, const void* A) {
  (void)K; (void)A;          // any K and alignment: the packing pre-pass has a scalar path
  return M >= 16;
}

int q4k_gemm(const char* op, const float* A, const uint8_t* W, void* C, int c_f16, int M, int N, int K,
             float alpha, const float* residual, const float* norm_weight, float norm_eps, int norm_weight_offset) {
  GemmArgs a{};
  a.A = A; a.W = W; a.W2 = nullptr; a.C = C; a.residual = residual;
  a.M = M; a.N = N; a.K = K; a.nb = (K + kQK - 1) / kQK;
  a.alpha = alpha; a.c_f16 = c_f16;
  a.norm_weight = norm_weight; a.norm_eps = norm_eps; a.norm_weight_offset = norm_weight_offset;
  return launch_gemm<false>(a, op);
}

int q4k_gemm_gate_up(const char* op, const float* A, const uint8_t* Wg, const uint8_t* Wu, float* C, int M,
                     int hidden, int inter, int activation, float alpha, float clamp_max,
                     const float* norm_weight, float norm_eps, int norm_weight_offset) {
  GemmArgs a{};
  a.A = A; a.W = Wg; a.W2 = Wu; a.C = C; a.residual = nullptr;
  a.M = M; a.N = inter; a.K = hidden; a.nb = (hidden + kQK - 1) / kQK;
  a.alpha = alpha; a.c_f16 = 0; a.activation = activation; a.clamp_max = clamp_max;
  a.norm_weight = norm_weight; a.norm_eps = norm_eps; a.norm_weight_offset = norm_weight_offset;
  return launch_gemm<true>(a, op);
}

}  // namespace dh

extern "C" int dh_q4k_gemm_layout(int M, int N, int K, int dual, int num_cus, int64_t* out4) {
  if (!out4 || M < 16 || N <= 0 || K <= 0) return 0;
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  const int wide = takes_wide(M, N, K, dual != 0) && choose_narrow(M, N, K, dual != 0).bm == 0 ? 1 : 0;
  const WideChoice pick = choose_wide(M, N, K, dual != 0);
  dh::plan_end();
  const int64_t steps = dh::ceil_div(K, BK);
  constexpr int rows_per_wave[] = {128, 128, 64, 64};
  const int64_t out[4] = {kWide[pick.tile].bm, kWide[pick.tile].rows, rows_per_wave[pick.tile], dh::ceil_div(steps, steps_per_piece(K, pick.pieces))};
  for (int i = 0; i < 4; i++) out4[i] = wide ? out[i] : 0;
  return wide;
}

extern "C" int dh_q4k_gemm_narrow_layout(int M, int N, int K, int dual, int num_cus, int64_t* out2) {
  if (!out2 || M < 16 || N <= 0 || K <= 0) return 0;
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  const NarrowChoice pick = choose_narrow(M, N, K, dual != 0);
  dh::plan_end();
  out2[0] = pick.bm;
  out2[1] = pick.bm ? dh::ceil_div(dh::ceil_div(K, BK), steps_per_piece(K, pick.pieces)) : 0;
  return pick.bm ? 1 : 0;
}
