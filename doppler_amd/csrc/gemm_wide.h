// Matrix products of 16-bit operands: operands from memory straight into LDS, v_mfma_f32_32x32x16 with f32 accumulation.
#pragma once
#include "dense_device.h"

namespace dh {

// WM x WN waves; a wave computes 64 FA rows x 64 FB columns as four quadrants of 32 FA x 32 FB.
template <int WM_, int WN_, int FA_, int FB_>
struct WideTile {
  static constexpr int WM = WM_, WN = WN_, FA = FA_, FB = FB_;
  static constexpr int BM = 64 * FA * WM, BN = 64 * FB * WN;
  static constexpr int kHalfA = BM / 2 * 128, kHalfB = BN / 2 * 128;       // bytes of half a tile's rows, 64 k
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kRound = 1024 * kWaves;                             // bytes all waves fetch with one load each: 8 rows a wave
  static constexpr int kRoundsA = kHalfA / kRound, kRoundsB = kHalfB / kRound;
  static constexpr int kAhead = BM * BN < 256 * 256 ? 4 : 0, kBegun = 2;                    // WeightLines; steps fetched in front of them
  static constexpr int kScratch = 4 * (kHalfA + kHalfB);
  static constexpr int kLds = kScratch + (kAhead ? 256 : 0);
  static_assert(kHalfA % kRound == 0 && kHalfB % kRound == 0, "whole loads");
};

typedef __attribute__((ext_vector_type(4))) uint32_t buffer_words_t;
__device__ __forceinline__ buffer_words_t buffer_words(const void* base) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return buffer_words_t{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p), (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32)),
                        0xffffffffu, 0x00020000u};
}
// 16 bytes per lane from base + v_off + s_off to LDS at lds + 16 * lane.  Inline assembly without register results: to the
// compiler the fetch does not exist, so its own LDS reads wait for no fetch in flight; the waits are written where the data is due.
// (s_nop: wait states between a vector instruction that writes a scalar operand, or the write of m0, and the fetch.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void fetch_to_lds(const buffer_words_t& words, uint32_t v_off, uint32_t s_off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(v_off), "s"(words), "s"(s_off)
               : "m0", "memory");
}
// The same from an address of its own per lane.
__device__ __forceinline__ void fetch_global_to_lds(const void* from, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(from) : "m0", "memory");
}
__device__ __forceinline__ void fetch_words_to_lds(const void* from, uint32_t lds) {      // 4 bytes per lane, to lds + 4 * lane
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(from) : "m0", "memory");
}
// 4 bytes per lane as in the first, to lds + 4 * lane.
__device__ __forceinline__ void touch_to_lds(const buffer_words_t& words, uint32_t v_off, uint32_t s_off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(v_off), "s"(words), "s"(s_off)
               : "m0", "memory");
}
#pragma clang diagnostic pop
// At most `fetches` of this wave's fetches still in flight, all its LDS reads done, then the other waves.
template <int fetches>
__device__ __forceinline__ void arrive_and_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(fetches) : "memory");
}

// The workgroups whose tiles lie in one stretch of columns read the same weights at about the same time.  Those come from HBM, about 1 us
// away, which the fetches of a tile below 256 x 256 are not far enough ahead for, and every one of the company then waits for the
// same lines.  So they take turns: at step t of every `count` one of them asks for a word of every line of step t + kAhead (64 lines a wave and
// instruction), which brings the line into the L2 of their die; the words land in 256 bytes of LDS that nobody reads.  us, weights from HBM:
// 1531 x 2048 x 6144 on 128 x 128 tiles 62 -> 51 (44 with weights that the 256 MB cache still holds), 1531 x 2048 x 3072 34 -> 27, 600 x 4096 x 4096
// 36 -> 32, 2048 x 4096 x 16384 on 256 x 128 264 -> 226, 300 x 6144 x 2048 on 64 x 64 19.2 -> 18.1.  Fewer than four tiles gain nothing (100 x 4096 x 12288
// on 64 x 64 54 -> 55), a 256 x 256 tile's step is longer than the way to HBM (47 -> 47.5), and activations asked for in the same way cost what
// they give (they are in the cache, having just been written).
// The waits below count fetches; a line asked for in between makes a wait reach one fetch further than it must, never less far.
struct Company {
  int index, count;
};
template <class Tile>
struct WeightLines {
  static constexpr int kLeast = 4;
  const buffer_words_t& words;
  uint32_t v_off, s_off, lds;
  int next, every, last;
  template <class OffW>
  __device__ __forceinline__ WeightLines(const buffer_words_t& ww, OffW w_off, uint32_t k_bytes, int nk, uint32_t lds0, int wave, int lane, Company c)
      : words(ww), v_off(w_off((wave % (Tile::BN / 64)) * 64 + lane)), s_off(k_bytes), lds(lds0 + Tile::kScratch),
        next(c.count >= kLeast && wave < Tile::BN / 64 ? c.index : -1), every(c.count), last(nk) {
    for (int t = next; (uint32_t)t < Tile::kAhead && t < last; t += every)
      if (t >= Tile::kBegun) touch_to_lds(words, v_off, s_off + 128u * (uint32_t)t, lds);      // (the tile itself has fetched those in front)
  }
  __device__ __forceinline__ void at(int t) {
    if (t != next) return;                   // (-1: never, and nothing to count: 16 steps of few rows take 0.2 us more with it)
    next += every;
    if (t + Tile::kAhead < last) touch_to_lds(words, v_off, s_off + 128u * (uint32_t)(t + Tile::kAhead), lds);
  }
};

// One tile.  a_off / w_off give the byte offset of a tile's row from the base (below 4 GB); rows of both operands hold nk * 64
// elements of k from there, 16-byte aligned.  Results: acc[i][j], 32 x 32 each, wave (wm, wn) at rows 64 FA wm, columns 64 FB wn.
//
// A k step (64 elements) is four phases, one per quadrant of the wave's tile: (A0,B0) (A0,B1) (A1,B1) (A1,B0), where A0, A1 are
// the halves of every wave's rows.  In a phase a wave multiplies fragments it read from LDS in the phase before, reads the next
// phase's, and fetches one half tile from memory into the quarter of LDS whose last reads the previous barrier closed:
//
//     phase   multiplies     reads       fetches
//       0     A0 B0 (t)      B1 (t)      B0 (t + 2)
//       1     A0 B1 (t)      A1 (t)      B1 (t + 2)
//       2     A1 B1 (t)      A0 (t + 1)  A1 (t + 2)
//       3     A1 B0 (t)      B0 (t + 1)  A0 (t + 3)
//
// so a fetch has six phases to arrive (its half tile is read in the seventh after it) and an LDS read one.  Waits count: loads
// complete in order, and what six phases fetch is fixed; past the last step the last one is fetched again and never used.
// LDS rows are 128 bytes; a row's 16-byte piece p lies at slot p ^ (row / 2 & 7), which spreads a half wave's fragment reads over all
// banks, and since a fetch writes 64 consecutive pieces, every lane fetches the piece that belongs there.
template <class Tile, bool F16, class OffA, class OffW>
__device__ __forceinline__ void wide_product(f32x16_t (&acc)[2 * Tile::FA][2 * Tile::FB], const void* a_base, OffA a_off, const void* w_base,
                                             OffW w_off, uint32_t k_bytes, int nk, char* smem, Company company) {
  constexpr int FA = Tile::FA, FB = Tile::FB, RA = Tile::kRoundsA, RB = Tile::kRoundsB, HA = Tile::kHalfA, HB = Tile::kHalfB;
  constexpr int kStep = 2 * (RA + RB);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / Tile::WN, wn = wave % Tile::WN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const buffer_words_t wa = buffer_words(a_base), ww = buffer_words(w_base);

  // fetches: round r of half h covers the next 8 rows of every wave; a half is every wave's 32 FA (FB) rows in turn
  uint32_t va[2][RA], vb[2][RB];
  const int frow_lane = 8 * wave + (lane >> 3);
  const uint32_t piece = 16 * ((lane & 7) ^ ((frow_lane >> 1) & 7));
#pragma unroll
  for (int h = 0; h < 2; h++) {
#pragma unroll
    for (int r = 0; r < RA; r++) {
      const int row = 8 * Tile::kWaves * r + frow_lane;
      va[h][r] = a_off(row / (32 * FA) * (64 * FA) + 32 * FA * h + row % (32 * FA)) + piece;
    }
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const int row = 8 * Tile::kWaves * r + frow_lane;
      vb[h][r] = w_off(row / (32 * FB) * (64 * FB) + 32 * FB * h + row % (32 * FB)) + piece;
    }
  }
  const uint32_t lds_a = lds0 + 1024 * wave, lds_b = lds0 + 4 * HA + 1024 * wave;
  auto at_k = [&](int t) { return k_bytes + 128u * (uint32_t)min(t, nk - 1); };
  auto fetch_a = [&](int h, int t, int buf) {
#pragma unroll
    for (int r = 0; r < RA; r++) fetch_to_lds(wa, va[h][r], at_k(t), lds_a + (2 * buf + h) * HA + Tile::kRound * r);
  };
  auto fetch_b = [&](int h, int t, int buf) {
#pragma unroll
    for (int r = 0; r < RB; r++) fetch_to_lds(ww, vb[h][r], at_k(t), lds_b + (2 * buf + h) * HB + Tile::kRound * r);
  };

  // fragment reads: lane l holds row l & 31, k 8 (l >> 5) .. + 7 of every 16
  const int frow = lane & 31;
  const char *ra[4], *rb[4];
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    const int at = frow * 128 + 16 * ((2 * ks + (lane >> 5)) ^ ((frow >> 1) & 7));
    ra[ks] = smem + at + wm * (32 * FA * 128);
    rb[ks] = smem + at + 4 * HA + wn * (32 * FB * 128);
  }
  u32x4_t fa[2][FA][4], fb[2][FB][4];
#define DH_READ_A(h_, buf_, f_, ks_) \
  fa[h_][f_][ks_] = *reinterpret_cast<const u32x4_t*>(ra[ks_] + (2 * (buf_) + (h_)) * HA + (f_) * 4096)
#define DH_READ_B(set_, h_, buf_, g_, ks_) \
  fb[set_][g_][ks_] = *reinterpret_cast<const u32x4_t*>(rb[ks_] + (2 * (buf_) + (h_)) * HB + (g_) * 4096)

#pragma unroll
  for (int i = 0; i < 2 * FA; i++)
#pragma unroll
    for (int j = 0; j < 2 * FB; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

  // multiplies quadrant (ah, bh) (B fragments in `set`); in front of its matrix-core instructions 1 .. n - 1 `between` is called
  auto multiply = [&](auto ah, auto bh, auto set, auto&& between) {
    int n = 0;
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
      for (int f = 0; f < FA; f++)
#pragma unroll
        for (int g = 0; g < FB; g++) {
          f32x16_t& c = acc[ah * FA + f][bh * FB + g];
          if constexpr (F16)
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, fa[ah][f][ks]), __builtin_bit_cast(f16x8_t, fb[set][g][ks]), c, 0, 0, 0);
          else
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fa[ah][f][ks]), __builtin_bit_cast(bf16x8_t, fb[set][g][ks]), c, 0, 0, 0);
          between(n++);
          __builtin_amdgcn_sched_barrier(0);
        }
  };
  // matrix-core instructions of a phase; the LDS reads go out behind the first half of them, so that the last has arrived when
  // the phase ends, the fetches behind the second
  constexpr int NM = 4 * FA * FB;
  auto first = [](int n, int reads) { return min(reads, 2 * n * reads / NM); };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;

  struct NoLines {
    __device__ __forceinline__ void at(int) {}
  };
  auto weight_lines = [&] {
    if constexpr (Tile::kAhead > 0) return WeightLines<Tile>(ww, w_off, k_bytes, nk, lds0, wave, lane, company);
    else return NoLines{};
  };
  auto step = [&](int t, auto parity, auto& lines) {
    lines.at(t);
    constexpr int P = decltype(parity)::value, Q = P ^ 1;
    using IP = std::integral_constant<int, P>;
    using IQ = std::integral_constant<int, Q>;
    multiply(I0{}, I0{}, IP{}, [&](int n) {
      if (n == NM / 2) fetch_b(0, t + 2, P);
#pragma unroll
      for (int i = first(n, 4 * FB); i < first(n + 1, 4 * FB); i++) DH_READ_B(Q, 1, P, i >> 2, i & 3);
    });
    arrive_and_wait<kStep + RA + RB>();    // A1 (t) is there
    multiply(I0{}, I1{}, IQ{}, [&](int n) {
      if (n == NM / 2) fetch_b(1, t + 2, P);
#pragma unroll
      for (int i = first(n, 4 * FA); i < first(n + 1, 4 * FA); i++) DH_READ_A(1, P, i >> 2, i & 3);
    });
    arrive_and_wait<kStep + 2 * RB>();     // A0 (t + 1)
    multiply(I1{}, I1{}, IQ{}, [&](int n) {
      if (n == NM / 2) fetch_a(1, t + 2, P);
#pragma unroll
      for (int i = first(n, 4 * FA); i < first(n + 1, 4 * FA); i++) DH_READ_A(0, Q, i >> 2, i & 3);
    });
    arrive_and_wait<kStep + RA + RB>();    // B0 (t + 1)
    multiply(I1{}, I0{}, IP{}, [&](int n) {
      if (n == NM / 2) fetch_a(0, t + 3, Q);
#pragma unroll
      for (int i = first(n, 4 * FB); i < first(n + 1, 4 * FB); i++) DH_READ_B(Q, 0, Q, i >> 2, i & 3);
    });
    arrive_and_wait<kStep + 2 * RA>();     // B1 (t + 1)
  };

  fetch_a(0, 0, 0);
  fetch_b(0, 0, 0);
  fetch_b(1, 0, 0);
  fetch_a(1, 0, 0);
  fetch_a(0, 1, 1);
  fetch_b(0, 1, 1);
  fetch_b(1, 1, 1);
  fetch_a(1, 1, 1);
  auto lines = weight_lines();
  arrive_and_wait<2 * kStep - RA - RB>();  // A0 (0), B0 (0)
#pragma unroll
  for (int i = 0; i < 4 * FA; i++) DH_READ_A(0, 0, i >> 2, i & 3);
#pragma unroll
  for (int i = 0; i < 4 * FB; i++) DH_READ_B(0, 0, 0, i >> 2, i & 3);
  arrive_and_wait<2 * kStep - RA - RB>();
  fetch_a(0, 2, 0);
  arrive_and_wait<kStep + 2 * RA>();       // B1 (0)
  int t = 0;
  for (; t + 2 <= nk; t += 2) {
    step(t, I0{}, lines);
    step(t + 1, I1{}, lines);
  }
  if (t < nk) step(t, I0{}, lines);
  // nothing may be in flight towards LDS when the workgroup ends, and the next tile starts from an idle LDS
  arrive_and_wait<0>();
#undef DH_READ_A
#undef DH_READ_B
}

// The small relative, for products whose tiles are too few to hide a step's latency: WM x WN waves of 32 rows x 32 G columns, four k
// steps in LDS, one barrier a step, fetches three steps ahead; a step is 4 G matrix-core instructions for a wave (0.21 us a step with few
// workgroups on the device, against 0.33 us for the 128 x 128 tile above).  Fetches, LDS layout and fragments as there.
template <int WM_, int WN_, int G_>
struct SmallTile {
  static constexpr int WM = WM_, WN = WN_, G = G_, FA = 0, FB = 0;
  static constexpr int BM = 32 * WM, BN = 32 * G * WN, kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kBufA = BM * 128, kBufB = BN * 128, kRoundsA = kBufA / (1024 * kWaves), kRoundsB = kBufB / (1024 * kWaves);
  static constexpr int kAhead = 8, kBegun = 3, kScratch = 4 * (kBufA + kBufB), kLds = kScratch + 256;      // WeightLines
  static_assert(kBufA % (1024 * kWaves) == 0 && kBufB % (1024 * kWaves) == 0 && 4 * kBufA <= 65536 && 4 * kBufB <= 65536, "whole loads");
};
template <class Tile, bool F16, class OffA, class OffW>
__device__ __forceinline__ void small_product(f32x16_t (&acc)[Tile::G], const void* a_base, OffA a_off, const void* w_base, OffW w_off, uint32_t k_bytes, int nk,
                                              char* smem, Company company) {
  constexpr int G = Tile::G, RA = Tile::kRoundsA, RB = Tile::kRoundsB, R = RA + RB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / Tile::WN, wn = wave % Tile::WN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const buffer_words_t wa = buffer_words(a_base), ww = buffer_words(w_base);
  uint32_t va[RA], vb[RB];
  const int row_lane = 8 * wave + (lane >> 3);
  const uint32_t piece = 16 * ((lane & 7) ^ ((row_lane >> 1) & 7));
#pragma unroll
  for (int r = 0; r < RA; r++) va[r] = a_off(8 * Tile::kWaves * r + row_lane) + piece;
#pragma unroll
  for (int r = 0; r < RB; r++) vb[r] = w_off(8 * Tile::kWaves * r + row_lane) + piece;
  const uint32_t lds_a = lds0 + 1024 * wave, lds_b = lds0 + 4 * Tile::kBufA + 1024 * wave;
  auto fetch = [&](int t, int buf) {
    const uint32_t k = k_bytes + 128u * (uint32_t)min(t, nk - 1);
#pragma unroll
    for (int r = 0; r < RA; r++) fetch_to_lds(wa, va[r], k, lds_a + buf * Tile::kBufA + 1024 * Tile::kWaves * r);
#pragma unroll
    for (int r = 0; r < RB; r++) fetch_to_lds(ww, vb[r], k, lds_b + buf * Tile::kBufB + 1024 * Tile::kWaves * r);
  };
  const int frow = lane & 31;
  const char *ra[4], *rb[4];
#pragma unroll
  for (int ks = 0; ks < 4; ks++) {
    const int at = frow * 128 + 16 * ((2 * ks + (lane >> 5)) ^ ((frow >> 1) & 7));
    ra[ks] = smem + at + wm * 4096;
    rb[ks] = smem + at + 4 * Tile::kBufA + wn * (G * 4096);
  }
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[g][e] = 0.f;
  fetch(0, 0);
  fetch(1, 1);
  fetch(2, 2);
  WeightLines<Tile> lines(ww, w_off, k_bytes, nk, lds0, wave, lane, company);
  auto step = [&](int t, auto buffer) {
    constexpr int B = decltype(buffer)::value;
    lines.at(t);
    arrive_and_wait<2 * R>();                // step t is there for all, and all have read step t - 1
    fetch(t + 3, (B + 3) & 3);
    u32x4_t fa[4], fb[4][G];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      fa[ks] = *reinterpret_cast<const u32x4_t*>(ra[ks] + B * Tile::kBufA);
#pragma unroll
      for (int g = 0; g < G; g++) fb[ks][g] = *reinterpret_cast<const u32x4_t*>(rb[ks] + B * Tile::kBufB + g * 4096);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
      for (int g = 0; g < G; g++) {
        if constexpr (F16)
          acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, fa[ks]), __builtin_bit_cast(f16x8_t, fb[ks][g]), acc[g], 0, 0, 0);
        else
          acc[g] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fa[ks]), __builtin_bit_cast(bf16x8_t, fb[ks][g]), acc[g], 0, 0, 0);
      }
  };
  for (int t = 0;; t += 4) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 >= nk) break;
    step(t + 1, std::integral_constant<int, 1>{});
    if (t + 2 >= nk) break;
    step(t + 2, std::integral_constant<int, 2>{});
    if (t + 3 >= nk) break;
    step(t + 3, std::integral_constant<int, 3>{});
    if (t + 4 >= nk) break;
  }
  arrive_and_wait<0>();                      // nothing may be in flight towards LDS when the workgroup ends
}

}  // namespace dh
