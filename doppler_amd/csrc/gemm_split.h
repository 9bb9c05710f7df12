// Matrix products of f32 activations and bf16 weights on the bf16 matrix cores, exact in every product.
#pragma once
#include "gemm_wide.h"

namespace dh {

// An f32 is the exact sum of three bf16: its upper 16 bits, those of what remains, and the rest (8 + 8 + 8 significand bits; what a
// subtraction leaves fits the next) - unless it has bits below bf16's smallest number, 2^-133, which only one below 2^-110 can have: then the rest's lower
// half is not zero, and `lost` collects that.  A product of two bf16 is exact in f32, so three bf16 instructions give what an f32 one gives of an
// activation and a bf16 weight, in 3 x 32 cycles for 16 k against 8 x 64.  Of a pair of values the words hold (first, second).
struct SplitWords {
  u32x4_t high, mid, low;
};
__device__ __forceinline__ SplitWords split_words(const f32x4_t& a, const f32x4_t& b, uint32_t& lost) {
  SplitWords s;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float x0 = i < 2 ? a[2 * i] : b[2 * i - 4], x1 = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    const float r0 = x0 - __uint_as_float(u0 & 0xffff0000u), r1 = x1 - __uint_as_float(u1 & 0xffff0000u);
    const uint32_t v0 = __float_as_uint(r0), v1 = __float_as_uint(r1);
    const float q0 = r0 - __uint_as_float(v0 & 0xffff0000u), q1 = r1 - __uint_as_float(v1 & 0xffff0000u);
    s.high[i] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    s.mid[i] = __builtin_amdgcn_perm(v1, v0, 0x07060302u);
    s.low[i] = __builtin_amdgcn_perm(__float_as_uint(q1), __float_as_uint(q0), 0x07060302u);
    lost |= __float_as_uint(q0) | __float_as_uint(q1);
  }
  return s;
}

// WM waves of 32 rows, each with NF blocks of 32 columns; KG groups of such waves share a step of 64 k (each takes 64 / KG of them) and
// add up their sums in LDS at the end; S steps in LDS.
template <int WM_, int NF_, int KG_, int S_, int PER_SIMD_>
struct SplitTile {
  static constexpr int WM = WM_, NF = NF_, KG = KG_, S = S_, kPerSimd = PER_SIMD_;
  static constexpr int BM = 32 * WM, BN = 32 * NF, kWaves = WM * KG, kThreads = 64 * kWaves;
  static constexpr int kBufA = BM * 256, kBufB = BN * 128, kRoundsA = kBufA / (1024 * kWaves), kRoundsB = kBufB / (1024 * kWaves);
  static constexpr int kSums = kWaves * NF * 4096, kShare = WM * NF * 4 / kWaves, kLds = S * (kBufA + kBufB) > kSums ? S * (kBufA + kBufB) : kSums;
  static_assert(kBufA % (1024 * kWaves) == 0 && kBufB % (1024 * kWaves) == 0 && kLds <= 163840, "whole loads");
  static_assert(kLds >= kSums + 4 * (kWaves + BM) && WM * NF * 4 % kWaves == 0, "a word a wave and a row behind the sums, whole shares");
};

// Where a group's sums lie when the loop is over: lane l's four are rows 32 wm + 8 q + 4 (l >> 5) + 0 .. 3 of column 32 j + (l & 31).
template <class Tile>
__device__ __forceinline__ f32x4_t* split_sums(char* smem, int kg, int wm, int j, int q) {
  return reinterpret_cast<f32x4_t*>(smem) + (((kg * Tile::WM + wm) * Tile::NF + j) * 4 + q) * 64;
}

// A wave's share of a tile's sums: groups of four rows and 32 columns, u-th at (wm, j, q) as above.
template <class Tile>
struct SumPlace {
  int wm, j, q;
  __device__ __forceinline__ SumPlace(int u) {
    const int at = (threadIdx.x >> 6) + Tile::kWaves * u;
    q = at & 3, j = (at >> 2) % Tile::NF, wm = (at >> 2) / Tile::NF;
  }
};
// Whether a sum of parts is the product's.  Not if it is not finite: the parts of an infinite value, and a part that is zero times an infinite
// weight, are no numbers where the product is infinite.  Nor if it is of up to 2^-80, which may consist of products of parts that f32 does not
// hold.
__device__ __forceinline__ bool sound_sum(float v) { return fabsf(v) <= 3.402823466e38f && (v == 0.f || fabsf(v) >= 0x1p-80f); }
// Adds up the groups' sums; whether all are sound.
template <class Tile>
__device__ __forceinline__ bool join_sums(f32x4_t (&sums)[Tile::kShare], char* smem) {
  bool sound = true;
#pragma unroll
  for (int u = 0; u < Tile::kShare; u++) {
    const SumPlace<Tile> at(u);
    sums[u] = split_sums<Tile>(smem, 0, at.wm, at.j, at.q)[threadIdx.x & 63];
#pragma unroll
    for (int g = 1; g < Tile::KG; g++) sums[u] += split_sums<Tile>(smem, g, at.wm, at.j, at.q)[threadIdx.x & 63];
#pragma unroll
    for (int e = 0; e < 4; e++) sound = sound && sound_sum(sums[u][e]);
  }
  return sound;
}
// Whether it holds for the whole workgroup.
template <class Tile>
__device__ __forceinline__ bool everywhere(bool here, char* smem) {
  int* const words = reinterpret_cast<int*>(smem + Tile::kSums);
  const int all = __builtin_amdgcn_ballot_w64(!here) == 0ull;
  if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = all;
  __syncthreads();
  int every = 1;
#pragma unroll
  for (int w = 0; w < Tile::kWaves; w++) every &= words[w];
  return __builtin_amdgcn_readfirstlane(every) != 0;
}

// A word for each of the tile's rows, not zero where a lane that has split some of it found the parts short of it (`whole` is split_product's).
// In place behind the next barrier.
template <class Tile>
__device__ __forceinline__ const int* short_rows(bool whole, char* smem) {
  int* const rows = reinterpret_cast<int*>(smem + Tile::kSums) + Tile::kWaves;
  for (int r = threadIdx.x; r < Tile::BM; r += Tile::kThreads) rows[r] = 0;
  __syncthreads();
  if (!whole) rows[32 * ((threadIdx.x >> 6) % Tile::WM) + (threadIdx.x & 31)] = 1;
  return rows;
}

// The same tile on v_mfma_f32_32x32x2_f32, operands from memory into registers: for a tile whose sums the parts do not give.  Waves take the
// rows and the share of k that they have in split_product, a lane four k at a time.  Bound by the instruction, 64 cycles for 2 k: a row that is
// no number takes a call of 600 x 18464 x 4096 from 280 to 700 us, infinite rows in every tile to 1230 (each such sum by a lane of its own: 1000
// and 90000).
template <class Tile, class OffA, class OffW>
__device__ __forceinline__ void exact_product(const void* a_base, OffA a_off, const void* w_base, OffW w_off, int nk, char* smem) {
  constexpr int NF = Tile::NF, KS = 4 / Tile::KG;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / Tile::WM, wm = wave % Tile::WM, row = lane & 31, half = lane >> 5;
  const char *pa = static_cast<const char*>(a_base) + a_off(32 * wm + row) + 64 * KS * kg + 16 * half, *pw[NF];
  f32x16_t acc[NF];
#pragma unroll
  for (int j = 0; j < NF; j++) {
    pw[j] = static_cast<const char*>(w_base) + w_off(32 * j + row) + 32 * KS * kg + 8 * half;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[j][e] = 0.f;
  }
#pragma unroll 1
  for (int t = 0; t < nk; t++) {
    f32x4_t fa[2 * KS];
    uint2 fw[2 * KS][NF];
#pragma unroll
    for (int s = 0; s < 2 * KS; s++) {
      fa[s] = *reinterpret_cast<const f32x4_t*>(pa + 256 * (int64_t)t + 32 * s);
#pragma unroll
      for (int j = 0; j < NF; j++) fw[s][j] = *reinterpret_cast<const uint2*>(pw[j] + 128 * (int64_t)t + 16 * s);
    }
#pragma unroll
    for (int s = 0; s < 2 * KS; s++)
#pragma unroll
      for (int j = 0; j < NF; j++) {
        const f32x4_t w = {bf16_low(fw[s][j].x), bf16_high(fw[s][j].x), bf16_low(fw[s][j].y), bf16_high(fw[s][j].y)};
#pragma unroll
        for (int e = 0; e < 4; e++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s][e], w[e], acc[j], 0, 0, 0);
      }
  }
#pragma unroll
  for (int j = 0; j < NF; j++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      split_sums<Tile>(smem, kg, wm, j, q)[lane] = f32x4_t{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
}

// One tile; operands, offsets and fetches as in gemm_wide.h, with 4-byte rows of A.  An A row's 64 k are 256 bytes whose 16-byte piece p
// lies at slot p ^ (row & 15); W rows as there.  Leaves every group's sums in LDS; whether the parts of what this lane has split are the whole.
template <class Tile, class OffA, class OffW>
__device__ __forceinline__ bool split_product(const void* a_base, OffA a_off, const void* w_base, OffW w_off, int nk, char* smem) {
  constexpr int NF = Tile::NF, KG = Tile::KG, S = Tile::S, RA = Tile::kRoundsA, RB = Tile::kRoundsB, KS = 4 / KG;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / Tile::WM, wm = wave % Tile::WM;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const buffer_words_t wa = buffer_words(a_base), ww = buffer_words(w_base);
  uint32_t va[RA], vb[RB];
#pragma unroll
  for (int r = 0; r < RA; r++) {
    const int row = 4 * (Tile::kWaves * r + wave) + (lane >> 4);
    va[r] = a_off(row) + 16 * ((lane & 15) ^ (row & 15));
  }
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const int row = 8 * (Tile::kWaves * r + wave) + (lane >> 3);
    vb[r] = w_off(row) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  const uint32_t lds_a = lds0 + 1024 * wave, lds_b = lds0 + S * Tile::kBufA + 1024 * wave;
  auto fetch = [&](int t, int buf) {
    const uint32_t k = (uint32_t)min(t, nk - 1);
#pragma unroll
    for (int r = 0; r < RA; r++) fetch_to_lds(wa, va[r], 256u * k, lds_a + buf * Tile::kBufA + 1024 * Tile::kWaves * r);
#pragma unroll
    for (int r = 0; r < RB; r++) fetch_to_lds(ww, vb[r], 128u * k, lds_b + buf * Tile::kBufB + 1024 * Tile::kWaves * r);
  };
  const int frow = lane & 31, half = lane >> 5;
  const char *ra[KS][2], *rb[KS];
#pragma unroll
  for (int i = 0; i < KS; i++) {
    const int ks = kg * KS + i;
#pragma unroll
    for (int e = 0; e < 2; e++) ra[i][e] = smem + (32 * wm + frow) * 256 + 16 * ((4 * ks + 2 * half + e) ^ (frow & 15));
    rb[i] = smem + S * Tile::kBufA + frow * 128 + 16 * ((2 * ks + half) ^ ((frow >> 1) & 7));
  }
  // what the mid and low parts add up to is kept apart: sums of the high parts are rounded once for 16 k, the others hardly at all
  f32x16_t acc[NF], rest[NF];
#pragma unroll
  for (int j = 0; j < NF; j++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[j][e] = rest[j][e] = 0.f;
  f32x4_t fa[2];
  u32x4_t fb[2][NF];
  SplitWords words[2];
  uint32_t lost = 0;
  auto read = [&](int i, int buf, int set) {
#pragma unroll
    for (int e = 0; e < 2; e++) fa[e] = *reinterpret_cast<const f32x4_t*>(ra[i][e] + buf * Tile::kBufA);
#pragma unroll
    for (int j = 0; j < NF; j++) fb[set][j] = *reinterpret_cast<const u32x4_t*>(rb[i] + buf * Tile::kBufB + j * 4096);
  };
  auto multiply = [&](const u32x4_t& part, int set, f32x16_t (&sum)[NF]) {
#pragma unroll
    for (int j = 0; j < NF; j++)
      sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, part), __builtin_bit_cast(bf16x8_t, fb[set][j]), sum[j], 0, 0, 0);
  };
  // a wave multiplies 16 k while it reads and splits the next; the last step reads itself again
  auto step = [&](int t, int u) {
    const int B = u % S;
#pragma unroll
    for (int i = 0; i < KS; i++) {
      const int cur = (u * KS + i) & 1, next = cur ^ 1;
      if (i == KS - 1) {
        arrive_and_wait<(S - 2) * (RA + RB)>();  // step t + 1 is there for all, and all have read step t
        fetch(t + S, B);
        read(0, (B + 1) % S, next);
      } else {
        read(i + 1, B, next);
      }
      multiply(words[cur].low, cur, rest);
      multiply(words[cur].mid, cur, rest);
      multiply(words[cur].high, cur, acc);
      words[next] = split_words(fa[0], fa[1], lost);
      __builtin_amdgcn_sched_group_barrier(0x008, NF, 0);
#pragma unroll
      for (int n = 0; n < 2 * NF; n++) {
        __builtin_amdgcn_sched_group_barrier(0x002, 56 / (2 * NF), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    }
  };
#pragma unroll
  for (int t = 0; t < S; t++) fetch(t, t);
  arrive_and_wait<(S - 1) * (RA + RB)>();
  read(0, 0, 0);
  words[0] = split_words(fa[0], fa[1], lost);
  constexpr int U = S * KS % 2 ? 2 * S : S;      // steps after which buffers and sets of registers repeat
  bool more = true;
  for (int t = 0; more; t += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (u && t + u >= nk) break;
      step(t + u, u);
    }
    more = t + U < nk;
  }
  arrive_and_wait<0>();                          // nothing in flight towards LDS, and every wave has read its last step
#pragma unroll
  for (int j = 0; j < NF; j++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      split_sums<Tile>(smem, kg, wm, j, q)[lane] = f32x4_t{acc[j][4 * q] + rest[j][4 * q], acc[j][4 * q + 1] + rest[j][4 * q + 1],
                                                           acc[j][4 * q + 2] + rest[j][4 * q + 2], acc[j][4 * q + 3] + rest[j][4 * q + 3]};
  __syncthreads();
  return (lost & 0xffffu) == 0u;
}

}  // namespace dh
