// Prefill attention (T query tokens at once) over an f16 KV cache with grouped-query heads, on the
// matrix cores: the flash-attention recurrence with v_mfma_f32_16x16x32_f16.
//
// A workgroup serves 64 QT query tokens of one head with two groups of four waves: wave w of a group owns QT groups of 16
// consecutive query rows, group 0 takes the even key tiles and group 1 the odd ones, and the groups' accumulators meet in
// LDS at the end.  Under a causal mask the last queries see many times the keys of the first: two groups on one tile halve that
// longest chain and keep two waves on every SIMD to its end, where two workgroups of four waves on a compute unit left the longer
// of them alone.  Long tiles are dispatched first; a head's tiles go to one of the eight L2 caches where the head count allows it.
//
// Key and value tiles go from memory straight into LDS (two buffers per group, one barrier per tile, the next tile in
// flight during the whole of this one), 16-byte pieces of a row permuted so that no fragment read meets a bank conflict; values are
// read transposed (ds_read_b64_tr_b16).  QT = 2 for prompts long enough to fill the compute units with 128-query tiles: every
// fragment a wave reads from LDS then feeds two matrix-core instructions.  Fragments are read six ahead of their use.
//
// Measured (us; before: one group staged through registers, V transposed on the way into LDS, fragments read as they were
// needed -> now): H 32/8, T 2048: 101 -> 61 (562 TFLOP/s); 16/8, 4096: 171 -> 96; 32/8, 8192: 1051 -> 605 (908
// TFLOP/s); 16/8, 512: 14.5 -> 11.2.  SPEC with distance bias, H 16/4, D 128: T 2048 90 -> 44, T 4096 276 -> 129, window 512 33 -> 29; 16 heads of 128 + 64 shared, T 2048: 91 -> 51.
// What is left at 128 queries a workgroup: 34% of the matrix cores' cycles and about as much other vector work (exponentials) in turns.
// Measured without gain: the groups half a tile apart (one at the products while the other is at its exponentials, two
// barriers a tile: 61 -> 59 us, but 51 -> 62 us with shared keys); fetches spread between the products (61 -> 65 us).
//
// Everything is computed transposed, so that the softmax statistics of a query live in the lanes
// that also hold its output column and nothing has to be shuffled between the two products:
//   S^T = K . Q^T   A = K rows from LDS (16 bytes of a key row per lane), B = Q^T from registers
//                   (scale folded in, rounded to f16).  D[key][q]: lane (q = l & 15, g = l >> 4)
//                   gets keys 16j + 4g + i (i < 4) of key subtile j.
//   softmax         per query = per lane column: maxima and sums over a lane's 16 values, the
//                   maxima then across the four lanes l, l+16, l+32, l+48 (lane-swap
//                   instructions), the sums only once after the last tile; fp32, online rescale.
//   O^T = V^T . P^T B = P^T is exactly the lane's own probabilities (k-slot (g, i') stands for
//                   key 16 (2 kb + i'/4) + 4g + i'%4 of 32-key block kb: a contraction index may be
//                   renumbered as long as both operands agree), A = V^T read from LDS in that same
//                   slot order by two transposing reads, 16 dims x 4 keys each.
// Causal tiles beyond the tile's last query are never visited.
// The SPEC form (dh_attn_spec_prefill) serves the attention of decoders without rotary positions: queries are read
// from stacked projection rows, every score loses r1 log2(1 + r2 (i - j)) (the distance bias in the softmax's own
// units), value heads may differ in size from key heads (both are padded to the template's sizes with zeros in
// LDS and registers), probabilities enter the second product as f16 high part + residual (22 bits), and the output is
// gated per head and written in the operand type of the product that reads it.  A head's key may end in elements that all
// heads of the token share (dh_attn_spec_prefill_shared): those come from rows of their own.
#include <algorithm>
#include <cfloat>
#include <cstdlib>

#include "attention_spec.h"
#include "dense_device.h"
#include "gemm_wide.h"

namespace {

typedef __attribute__((ext_vector_type(8))) _Float16 half8_t;
typedef __attribute__((ext_vector_type(4))) float float4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;   // plain vector type: arrays of it stay in registers

// A 16-byte piece's slot in its row of LDS, and back.  Keys: a fragment read takes one piece of 16 rows, and the slots of
// those rows cover all banks (rows of an odd number of 128 bytes alternate between the banks' halves by themselves).  Values: pairs of
// pieces (the 16 elements of a transposing read) stay together.
template <int D>
__device__ __forceinline__ int swizzled_k(int row, int c) { return D / 64 % 2 ? c ^ ((row >> 1) & 7) : c ^ (row & 15); }
template <int VD>
__device__ __forceinline__ int swizzled_v(int row, int c) { return VD / 64 % 2 ? c ^ (2 * ((row >> 1) & 3)) : c ^ (2 * (row & 7)); }

typedef __attribute__((ext_vector_type(4))) _Float16 half4_t;
typedef __attribute__((ext_vector_type(4))) short short4_t;
__device__ __forceinline__ half4_t read_transposed(const char* p) {
  return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)p));
}

// The four lanes l, l ^ 16, l ^ 32, l ^ 48 hold one query's scores.  v_permlane32_swap and
// v_permlane16_swap (gfx950) hand a lane its partner's value through the vector ALU: with both
// operands the same register, one result holds the lane's own half (row) pair and the other the
// partner's.  No LDS round trip, and no wait that would also stall on outstanding fragment reads.
__device__ __forceinline__ float quad_rows_max(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quad_rows_sum(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

struct PrefillArgs {
  const float* Q;       // [T][H][D]
  const __half* K;      // [rows][Hkv][D]
  const __half* V;
  float* O;             // [T][H][D]
  int T, H, Hkv, G, kv_len, start_pos, causal, window;
  float scale, softcap;
  // ---- SPEC form only
  int dk, dv;           // head sizes of caches and projection rows (<= the template's, multiples of 8)
  int own_k;            // key elements of the head itself; the other dk - own_k are shared by all heads
  const __half* KS;     // their rows, ld_shared apart
  int64_t ld_shared;
  int64_t ld_q, ld_o;
  const float* r1;      // [H] or null
  const float* r2;
  const float* gate;    // H numbers per query token, ld_q apart, or null
  uint16_t* O16;        // bf16 output instead of O
};

// Four elements of an output row in the type of the product that reads it.
__device__ __forceinline__ void store_spec(const PrefillArgs& a, int64_t at, float4_t v) {
  if (a.O16) {
    uint2 two;
    two.x = (uint32_t)dh::f32_to_bf16_bits(v[0]) | ((uint32_t)dh::f32_to_bf16_bits(v[1]) << 16);
    two.y = (uint32_t)dh::f32_to_bf16_bits(v[2]) | ((uint32_t)dh::f32_to_bf16_bits(v[3]) << 16);
    *reinterpret_cast<uint2*>(a.O16 + at) = two;
  } else {
    *reinterpret_cast<float4*>(a.O + at) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

template <int D, int VD, int QT, bool SPEC>
__global__ __launch_bounds__(512, 2) void attn_prefill_kernel(const PrefillArgs a) {
  constexpr int BQ = 64 * QT;
  constexpr int BKEYS = D > 192 ? 32 : 64;      // keys of a tile: four tiles (two groups, two buffers) in 160 KB of LDS
  constexpr int NJ = BKEYS / 16, NKB = BKEYS / 32;
  constexpr int STEPS = D / 32;            // MFMAs per 16 x 16 score tile
  constexpr int DT = VD / 16;              // output row tiles (of O^T)
  constexpr int AHEAD = 6;                 // fragments on their way from LDS
  constexpr int PIECES = BKEYS * D / 8 / 256;   // 16-byte pieces of a K tile per thread of a group
  constexpr int VPIECES = BKEYS * VD / 8 / 256;
  constexpr int KBYTES = BKEYS * D * 2, TILE = KBYTES + BKEYS * VD * 2;
  constexpr int MERGE_BYTES = 4 * QT * (DT * 1024 + 512);        // four waves' accumulators, maxima and sums
  static_assert(PIECES >= 1 && VPIECES >= 1 && MERGE_BYTES <= 4 * TILE && 4 * TILE <= 160 * 1024, "LDS");
  __shared__ __align__(1024) char smem[4 * TILE];

  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int tid = threadIdx.x & 255, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int q = lane & 15, g = lane >> 4;
  // late queries first, heads fastest; workgroups go round the eight XCDs, which get H / 8 neighbouring heads each
  const int id = blockIdx.y * gridDim.x + blockIdx.x;
  const int q0 = ((int)gridDim.x - 1 - id / a.H) * BQ;
  int h = id % a.H;
  if (a.H % 8 == 0) h = (h & 7) * (a.H / 8) + (h >> 3);
  const int kvh = h / a.G;
  const int dk = SPEC ? a.dk : D, dv = SPEC ? a.dv : VD;
  const int own_k = SPEC ? a.own_k : D;
  const int64_t k_stride = (int64_t)a.Hkv * own_k, v_stride = (int64_t)a.Hkv * dv;
  int my_q[QT], my_pos[QT];                                   // query token of this lane's column, its absolute position
#pragma unroll
  for (int u = 0; u < QT; u++) {
    my_q[u] = q0 + 16 * (QT * wave + u) + q;
    my_pos[u] = a.start_pos + my_q[u];
  }

  // ---- Q^T fragments (B operand): b[i] = scale * Q[my_q][32 s + 8 g + i].  Scores are kept in
  // units of log2(e), so that the softmax needs v_exp_f32 alone (with a soft cap the factor is
  // applied after the cap instead).
  constexpr float kLog2e = 1.4426950408889634f;
  const float qscale = a.softcap > 0.f ? a.scale : a.scale * kLog2e;
  half8_t qb[QT][STEPS];
#pragma unroll
  for (int u = 0; u < QT; u++)
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      const int64_t qrow = min(my_q[u], a.T - 1);
      const float* qp = a.Q + (SPEC ? qrow * a.ld_q + (int64_t)h * dk : (qrow * a.H + h) * D) + 32 * s + 8 * g;
      float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
      if (!SPEC || 32 * s + 8 * g < dk) { v0 = reinterpret_cast<const float4*>(qp)[0]; v1 = reinterpret_cast<const float4*>(qp)[1]; }
      const float qv[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
      for (int i = 0; i < 8; i++) qb[u][s][i] = (_Float16)(qv[i] * qscale);
    }

  // ---- key range of this query tile
  const int last_q = min(q0 + BQ, a.T) - 1;
  int kend = a.kv_len;
  if (a.causal) kend = min(kend, a.start_pos + last_q + 1);
  int kbeg = 0;
  if (a.window > 0) kbeg = max(0, a.start_pos + q0 - a.window + 1);
  kbeg = kbeg / BKEYS * BKEYS;
  const int ntiles = (kend - kbeg + BKEYS - 1) / BKEYS;

  float r1 = 0.f, r2 = 0.f;
  if (SPEC && a.r1) {
    r1 = a.r1[h];
    r2 = a.r2[h];
  }
  float4_t acc[QT][DT];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int u = 0; u < QT; u++) {
#pragma unroll
    for (int t = 0; t < DT; t++) acc[u][t] = {0.f, 0.f, 0.f, 0.f};
    m_run[u] = -FLT_MAX;
    l_run[u] = 0.f;
  }

  // ---- fetches: piece tid + 256 r of a tile's slots in LDS is loaded from where the swizzle says it belongs
  uint32_t k_at[PIECES], v_at[VPIECES];
  auto k_piece = [&](int r, int* row) { *row = (tid + 256 * r) / (D / 8); return swizzled_k<D>(*row, (tid + 256 * r) % (D / 8)); };
  auto v_piece = [&](int r, int* row) { *row = (tid + 256 * r) / (VD / 8); return swizzled_v<VD>(*row, (tid + 256 * r) % (VD / 8)); };
  const uint32_t k_row = 2 * (uint32_t)k_stride, s_row = SPEC ? 2 * (uint32_t)a.ld_shared : 0u, v_row = 2 * (uint32_t)v_stride;
  auto place = [&](int last) {                       // byte offsets of this lane's pieces in a tile whose last row is `last`
#pragma unroll
    for (int r = 0; r < PIECES; r++) {
      int row;
      const int c = k_piece(r, &row);
      k_at[r] = SPEC && 8 * c >= own_k ? min(row, last) * s_row + 2u * (8 * c - own_k) : min(row, last) * k_row + 16u * c;
    }
#pragma unroll
    for (int r = 0; r < VPIECES; r++) {
      int row;
      const int c = v_piece(r, &row);
      v_at[r] = min(row, last) * v_row + 16u * c;
    }
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + 1024u * wave;
  auto fetch = [&](int kt, int buf) {
    const int first = kbeg + kt * BKEYS;
    if (first + BKEYS > a.kv_len) place(a.kv_len - 1 - first);
    const uint32_t to = lds0 + (uint32_t)((2 * grp + buf) * TILE);
    const dh::buffer_words_t wk = dh::buffer_words(a.K + (int64_t)first * k_stride + (int64_t)kvh * own_k);
    const dh::buffer_words_t wv = dh::buffer_words(a.V + (int64_t)first * v_stride + (int64_t)kvh * dv);
#pragma unroll
    for (int r = 0; r < PIECES; r++) {
      int row;
      const int c = k_piece(r, &row);
      if (!SPEC || 8 * c < own_k) {
        dh::fetch_to_lds(wk, k_at[r], 0, to + 4096u * r);
      } else if (8 * c < dk) {
        dh::fetch_to_lds(dh::buffer_words(a.KS + (int64_t)first * a.ld_shared), k_at[r], 0, to + 4096u * r);
      }
    }
#pragma unroll
    for (int r = 0; r < VPIECES; r++) {
      int row;
      const int c = v_piece(r, &row);
      if (!SPEC || 8 * c < dv) dh::fetch_to_lds(wv, v_at[r], 0, to + KBYTES + 4096u * r);
    }
  };
  if (SPEC) {                                        // elements beyond the heads' sizes: nothing is fetched there
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    for (int buf = 0; buf < 2; buf++) {
      char* to = smem + (2 * grp + buf) * TILE + 16 * tid;
#pragma unroll
      for (int r = 0; r < PIECES; r++) {
        int row;
        if (8 * k_piece(r, &row) >= dk) *reinterpret_cast<u32x4_t*>(to + 4096 * r) = zero;
      }
#pragma unroll
      for (int r = 0; r < VPIECES; r++) {
        int row;
        if (8 * v_piece(r, &row) >= dv) *reinterpret_cast<u32x4_t*>(to + KBYTES + 4096 * r) = zero;
      }
    }
  }
  place(BKEYS - 1);
  if (grp < ntiles) fetch(grp, 0);

  // fragment addresses in a tile: the swizzles depend on the lane alone, so a step is an exclusive or, a row block an offset
  const int k_lane = q * (2 * D) + 16 * swizzled_k<D>(q, g);
  const int v_lane = KBYTES + (4 * g + (q >> 2)) * (2 * VD) + 16 * swizzled_v<VD>(4 * g + (q >> 2), (q & 3) >> 1) + 8 * (q & 1);
  for (int it = 0; 2 * it < ntiles; it++) {
    const int kt = 2 * it + grp;
    dh::arrive_and_wait<0>();                          // the tile is there, and the other buffer read by all
    if (kt + 2 < ntiles) fetch(kt + 2, (it + 1) & 1);
    if (kt >= ntiles) continue;

    // ---- S^T for this wave's 16 QT queries against the 64 keys
    const int kbase = kbeg + kt * BKEYS;
    if (a.causal && kbase > a.start_pos + q0 + 16 * QT * (wave + 1) - 1) continue;    // behind all of the wave's queries
    float4_t st[QT][NJ];
    half8_t ring[AHEAD];
    const int at = (2 * grp + (it & 1)) * TILE;
    auto k_fragment = [&](int f) {
      constexpr int X = D / 64 % 2 ? 1 : 3;            // steps inside the swizzled part of a row
      const int j = f % NJ, step = f / NJ;
      return *reinterpret_cast<const half8_t*>(smem + (((at + k_lane) ^ (64 * (step & X))) + 64 * (step & ~X) + 32 * D * j));
    };
    auto v_fragment = [&](int f) {
      const int t = f % DT, kb = f / DT;
      const char* p = smem + (((at + v_lane) ^ (32 * t)) + 64 * VD * kb);
      const half4_t lo = read_transposed(p), hi = read_transposed(p + 32 * VD);
      return half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
#pragma unroll
    for (int f = 0; f < AHEAD; f++) ring[f] = k_fragment(f);
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int u = 0; u < QT; u++) st[u][j] = {0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < NJ * STEPS; f++) {
#pragma unroll
      for (int u = 0; u < QT; u++) st[u][f % NJ] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[f % AHEAD], qb[u][f / NJ], st[u][f % NJ], 0, 0, 0);
      if (f + AHEAD < NJ * STEPS) ring[f % AHEAD] = k_fragment(f + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < AHEAD; f++) ring[f] = v_fragment(f);
    __builtin_amdgcn_sched_barrier(0);
    // ---- mask, soft cap, online softmax (this lane: query my_q, keys kbase + 16 j + 4 g + i).
    // A tile that every query of a 16-query group sees completely needs no per-element masks.
    half8_t pb[QT][NKB];
    half8_t pl[SPEC ? QT : 1][NKB];            // SPEC: what the f16 probabilities left over
    float alpha[QT];
    bool rescale = false;
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const int grp_lo = a.start_pos + q0 + 16 * (QT * wave + u), grp_hi = grp_lo + 15;
      const bool full = kbase + BKEYS <= a.kv_len && (!a.causal || kbase + BKEYS - 1 <= grp_lo) &&
                        (a.window <= 0 || kbase > grp_hi - a.window);
      float mx = -FLT_MAX;
      if (SPEC && a.r1) {
        const float d0 = (float)(my_pos[u] - kbase - 4 * g);
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int i = 0; i < 4; i++)         // keys behind the query give NaN or less; they are masked below
            st[u][j][i] = fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, d0 - (float)(16 * j + i), 1.0f)), st[u][j][i]);
      }
      if (a.softcap > 0.f) {
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int i = 0; i < 4; i++) st[u][j][i] = tanhf(st[u][j][i] / a.softcap) * (a.softcap * kLog2e);
      }
      if (!full) {                            // this lane's keys are 16 j + i behind kbase + 4 g
        const int last = min(a.causal ? my_pos[u] : a.kv_len - 1, a.kv_len - 1) - kbase - 4 * g;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int i = 0; i < 4; i++) st[u][j][i] = 16 * j + i <= last ? st[u][j][i] : -INFINITY;
        if (a.window > 0) {
          const int first = my_pos[u] - a.window + 1 - kbase - 4 * g;
#pragma unroll
          for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) st[u][j][i] = 16 * j + i >= first ? st[u][j][i] : -INFINITY;
        }
      }
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) mx = fmaxf(mx, st[u][j][i]);
      mx = quad_rows_max(mx);
      // m_run need not be the maximum, only near it: up to 2^8 the probabilities keep their precision in f16, and the
      // accumulators are scaled seldom.  Finite: it starts at -FLT_MAX.
      const float m_new = mx > m_run[u] + 8.f ? mx : m_run[u];
      alpha[u] = __builtin_amdgcn_exp2f(m_run[u] - m_new);
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float p = __builtin_amdgcn_exp2f(st[u][j][i] - m_new);   // 2^-inf = 0 for masked keys
          ps += p;
          const _Float16 ph = (_Float16)p;
          pb[u][j >> 1][4 * (j & 1) + i] = ph;
          if constexpr (SPEC) pl[u][j >> 1][4 * (j & 1) + i] = (_Float16)(p - (float)ph);
        }
      l_run[u] = l_run[u] * alpha[u] + ps;               // this lane's share: alpha is the query's, the sum is taken once at the end
      m_run[u] = m_new;
      rescale = rescale || __builtin_amdgcn_ballot_w64(alpha[u] != 1.0f) != 0;   // else nothing to scale
    }
    // ---- O^T = alpha O^T + V^T P^T
    if (rescale) {
#pragma unroll
      for (int t = 0; t < DT; t++)
#pragma unroll
        for (int u = 0; u < QT; u++) acc[u][t] *= alpha[u];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < NKB * DT; f++) {
      const int t = f % DT, kb = f / DT;
#pragma unroll
      for (int u = 0; u < QT; u++) acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[f % AHEAD], pb[u][kb], acc[u][t], 0, 0, 0);
      if constexpr (SPEC) {
#pragma unroll
        for (int u = 0; u < QT; u++) acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[f % AHEAD], pl[u][kb], acc[u][t], 0, 0, 0);
      }
      if (f + AHEAD < NKB * DT) ring[f % AHEAD] = v_fragment(f + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- the two groups' shares of a query, through LDS; a single tile is group 0's alone (prompts of 64 tokens, D 128: 6.2 -> 5.7 us)
  if (ntiles > 1) {
    __syncthreads();
    float4_t* shared_acc = reinterpret_cast<float4_t*>(smem) + wave * (QT * DT * 64) + lane;
    float2* shared_ml = reinterpret_cast<float2*>(smem + 4 * QT * DT * 1024) + wave * (QT * 64) + lane;
    if (grp) {
#pragma unroll
      for (int u = 0; u < QT; u++) {
#pragma unroll
        for (int t = 0; t < DT; t++) shared_acc[64 * (u * DT + t)] = acc[u][t];
        shared_ml[64 * u] = make_float2(m_run[u], l_run[u]);
      }
    }
    __syncthreads();
    if (!grp) {
#pragma unroll
      for (int u = 0; u < QT; u++) {
        const float2 ml = shared_ml[64 * u];
        const float m = fmaxf(m_run[u], ml.x), mine = __builtin_amdgcn_exp2f(m_run[u] - m), other = __builtin_amdgcn_exp2f(ml.x - m);
        l_run[u] = l_run[u] * mine + ml.y * other;
#pragma unroll
        for (int t = 0; t < DT; t++) acc[u][t] = acc[u][t] * mine + shared_acc[64 * (u * DT + t)] * other;
      }
    }
  }
  if (grp) return;

  // ---- lane (q, g) holds O[my_q][16 t + 4 g + i]
#pragma unroll
  for (int u = 0; u < QT; u++) {
    const float l = quad_rows_sum(l_run[u]);
    if (my_q[u] < a.T) {
      float inv = l > 0.f ? 1.0f / l : 0.f;
      if constexpr (SPEC) {
        if (a.gate) inv *= 1.0f / (1.0f + expf(-a.gate[(int64_t)my_q[u] * a.ld_q + h]));
        const int64_t at = (int64_t)my_q[u] * a.ld_o + (int64_t)h * dv + 4 * g;
#pragma unroll
        for (int t = 0; t < DT; t++) {
          if (16 * t + 4 * g >= dv) continue;
          store_spec(a, at + 16 * t, acc[u][t] * inv);
        }
        continue;
      }
      float* op = a.O + ((int64_t)my_q[u] * a.H + h) * D + 4 * g;
#pragma unroll
      for (int t = 0; t < DT; t++)
        *reinterpret_cast<float4*>(op + 16 * t) =
            make_float4(acc[u][t][0] * inv, acc[u][t][1] * inv, acc[u][t][2] * inv, acc[u][t][3] * inv);
    }
  }
}

// The same over a 32-bit cache, everything in 32 bits (v_mfma_f32_16x16x4_f32; a lane's four consecutive elements of a key row feed
// four instructions, whose k-slot g stands for element 4 g + e on both sides).  A workgroup is eight waves on the same
// 16 queries of a head; a wave takes every eighth tile of 32 keys, straight from memory into registers (values requested before the
// scores are computed, the next keys before the exponentials), and the waves meet in LDS at the end.  The general kernel reads every
// key again for each query: us, H 16/8, D 64, before -> now: T 301 28 -> 11, T 1024 164 -> 52, T 4096 1926 -> 549 (63 of 136 TFLOP/s;
// each workgroup reads its keys from L2 on its own); D 128, window 1024, T 2048 845 -> 251.
template <int D, int VD>
__global__ __launch_bounds__(512) void attn_prefill_f32_kernel(const PrefillArgs a) {
  constexpr int WAVES = 8, STEPS = D / 16, DT = VD / 16, BKEYS = 32;
  __shared__ __align__(16) float4_t acc_s[WAVES][DT][64];
  __shared__ float2 ml_s[WAVES][16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int q = lane & 15, g = lane >> 4;
  const int id = blockIdx.y * gridDim.x + blockIdx.x;            // late queries first
  const int q0 = ((int)gridDim.x - 1 - id / a.H) * 16, h = id % a.H, kvh = h / a.G;
  const int my_q = q0 + q, my_pos = a.start_pos + my_q;
  const float* K = reinterpret_cast<const float*>(a.K) + (int64_t)kvh * a.own_k;
  const float* V = reinterpret_cast<const float*>(a.V) + (int64_t)kvh * a.dv;
  const float* KS = reinterpret_cast<const float*>(a.KS);
  const int64_t k_stride = (int64_t)a.Hkv * a.own_k, v_stride = (int64_t)a.Hkv * a.dv;
  const int kend = min(a.kv_len, a.start_pos + min(q0 + 16, a.T));
  const int kbeg = a.window > 0 ? max(0, a.start_pos + q0 - a.window + 1) / BKEYS * BKEYS : 0;
  const int ntiles = (kend - kbeg + BKEYS - 1) / BKEYS;

  float4_t kf[2][STEPS], qb[STEPS];
  float vf[8][DT];
  auto load_k = [&](int kt) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int64_t row = min(kbeg + kt * BKEYS + 16 * j + q, a.kv_len - 1);
#pragma unroll
      for (int s = 0; s < STEPS; s++) {
        const int dim = 16 * s + 4 * g;
        kf[j][s] = float4_t{0.f, 0.f, 0.f, 0.f};
        if (dim < a.own_k) kf[j][s] = *reinterpret_cast<const float4_t*>(K + row * k_stride + dim);
        else if (dim < a.dk) kf[j][s] = *reinterpret_cast<const float4_t*>(KS + row * a.ld_shared + dim - a.own_k);
      }
    }
  };
  if (wave < ntiles) load_k(wave);
  const float* qp = a.Q + (int64_t)min(my_q, a.T - 1) * a.ld_q + (int64_t)h * a.dk + 4 * g;
  constexpr float kLog2e = 1.4426950408889634f;
#pragma unroll
  for (int s = 0; s < STEPS; s++) {
    qb[s] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (16 * s + 4 * g < a.dk) qb[s] = *reinterpret_cast<const float4_t*>(qp + 16 * s) * (a.scale * kLog2e);
  }
  float r1 = 0.f, r2 = 0.f;
  if (a.r1) {
    r1 = a.r1[h];
    r2 = a.r2[h];
  }
  float4_t acc[DT];
#pragma unroll
  for (int t = 0; t < DT; t++) acc[t] = {0.f, 0.f, 0.f, 0.f};
  float m_run = -FLT_MAX, l_run = 0.f;
  bool left_out = false;
  auto in_part = [&](int kbase) { return kbase + BKEYS - 1 > a.start_pos + q0 || (a.window > 0 && kbase + a.window < a.start_pos + q0 + 16); };
  for (int kt = wave; kt < ntiles; kt += WAVES) {
    const int kbase = kbeg + kt * BKEYS;
#pragma unroll
    for (int n = 0; n < 8; n++) {
      const int64_t row = min(kbase + 16 * (n >> 2) + 4 * g + (n & 3), a.kv_len - 1);
#pragma unroll
      for (int t = 0; t < DT; t++) vf[n][t] = 16 * t + q < a.dv ? V[row * v_stride + 16 * t + q] : 0.f;
    }
    float4_t st[2];
#pragma unroll
    for (int j = 0; j < 2; j++) st[j] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STEPS; s++)
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int j = 0; j < 2; j++) st[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][s][e], qb[s][e], st[j], 0, 0, 0);
    if (kt + WAVES < ntiles) load_k(kt + WAVES);
    const float d0 = (float)(my_pos - kbase - 4 * g);
    const int last = min(my_pos, a.kv_len - 1) - kbase - 4 * g, first = a.window > 0 ? my_pos - a.window + 1 - kbase - 4 * g : -BKEYS;
    float mx = -FLT_MAX;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {           // keys behind the query give NaN or less; they are masked
        float v = st[j][i];
        if (a.r1) v = fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, d0 - (float)(16 * j + i), 1.0f)), v);
        v = 16 * j + i <= last && 16 * j + i >= first ? v : -INFINITY;
        st[j][i] = v;
        mx = fmaxf(mx, v);
      }
    const float m_new = fmaxf(m_run, quad_rows_max(mx));         // finite: m_run starts at -FLT_MAX
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    float ps = 0.f;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        st[j][i] = __builtin_amdgcn_exp2f(st[j][i] - m_new);     // 2^-inf = 0 for masked keys
        ps += st[j][i];
      }
    l_run = l_run * alpha + ps;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < DT; t++) acc[t] *= alpha;
    // Where not every query sees the whole tile, values that are not finite count as zero here (a masked probability of 0 would make
    // them NaN); the queries that see them get them behind the loop.
    if (in_part(kbase)) {
      float z = 0.f;
#pragma unroll
      for (int n = 0; n < 8; n++)
#pragma unroll
        for (int t = 0; t < DT; t++) z = fmaf(vf[n][t], 0.f, z);
      if (__builtin_amdgcn_ballot_w64(!(z == 0.f))) {
        left_out = true;
#pragma unroll
        for (int n = 0; n < 8; n++)
#pragma unroll
          for (int t = 0; t < DT; t++) vf[n][t] = fabsf(vf[n][t]) < INFINITY ? vf[n][t] : 0.f;
      }
    }
#pragma unroll
    for (int n = 0; n < 8; n++)
#pragma unroll
      for (int t = 0; t < DT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[n][t], st[n >> 2][n & 3], acc[t], 0, 0, 0);
  }
  // The lane's place once more, from the hardware: kept through the loop it would cost the registers of the largest form (128, 128) that
  // the loop needs (addresses spilled, 248 -> 267 us at T 2048).
  const int out_lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), out_g = out_lane >> 4;
  const int out_q = q0 + (out_lane & 15), out_pos = a.start_pos + out_q;
  if (left_out) {
    for (int kt = wave; kt < ntiles; kt += WAVES) {
      if (!in_part(kbeg + kt * BKEYS)) continue;
      const int last = min(kbeg + (kt + 1) * BKEYS - 1, min(out_pos, a.kv_len - 1));
      for (int key = max(kbeg + kt * BKEYS, a.window > 0 ? out_pos - a.window + 1 : 0); key <= last; key++)
#pragma unroll
        for (int t = 0; t < DT; t++) {
          if (16 * t + 4 * out_g >= a.dv) continue;
          const float4_t v = *reinterpret_cast<const float4_t*>(V + key * v_stride + 16 * t + 4 * out_g);
#pragma unroll
          for (int e = 0; e < 4; e++) acc[t][e] = fabsf(v[e]) < INFINITY ? acc[t][e] : acc[t][e] + v[e];
        }
    }
  }
#pragma unroll
  for (int t = 0; t < DT; t++) acc_s[wave][t][out_lane] = acc[t];
  l_run = quad_rows_sum(l_run);
  if (out_g == 0) ml_s[wave][out_lane & 15] = make_float2(m_run, l_run);
  __syncthreads();
  if (out_q >= a.T) return;
  float m = -FLT_MAX, l = 0.f, part[WAVES];
#pragma unroll
  for (int w = 0; w < WAVES; w++) m = fmaxf(m, ml_s[w][out_lane & 15].x);
#pragma unroll
  for (int w = 0; w < WAVES; w++) {
    part[w] = __builtin_amdgcn_exp2f(ml_s[w][out_lane & 15].x - m);
    l = fmaf(part[w], ml_s[w][out_lane & 15].y, l);
  }
  float inv = l > 0.f ? 1.0f / l : 0.f;
  if (a.gate) inv *= 1.0f / (1.0f + expf(-a.gate[(int64_t)out_q * a.ld_q + h]));
  const int64_t at = (int64_t)out_q * a.ld_o + (int64_t)h * a.dv + 4 * out_g;
  for (int t = wave; t < DT; t += WAVES) {
    if (16 * t + 4 * out_g >= a.dv) continue;
    float4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < WAVES; w++) o += acc_s[w][t][out_lane] * part[w];
    store_spec(a, at + 16 * t, o * inv);
  }
}

}  // namespace

extern "C" int dh_attn_prefill(const float* d_Q, const void* d_K, const void* d_V, float* d_O, int T, int H,
                               int Hkv, int D, int kv_len, float scale, int causal, int start_pos,
                               float softcap, int sliding_window) {
  const char* op = "dh_attn_prefill";
  DH_REQUIRE_INIT(op);
  if (T <= 0 || H <= 0 || Hkv <= 0 || D <= 0)
    return dh::fail(1, "[%s] seqLen/numHeads/numKVHeads/headDim must be positive", op);
  if (H % Hkv) return dh::fail(1, "[%s] numHeads=%d must be a multiple of numKVHeads=%d", op, H, Hkv);
  if (D != 64 && D != 128) return dh::fail(1, "[%s] headDim %d not supported (64, 128)", op, D);
  if (kv_len <= 0 || start_pos < 0 || sliding_window < 0)
    return dh::fail(1, "[%s] kvLen must be positive, startPos and slidingWindow non-negative", op);
  if (causal && start_pos + T > kv_len)
    return dh::fail(1, "[%s] startPos=%d + seqLen=%d exceeds kvLen=%d", op, start_pos, T, kv_len);
  if (!d_Q || !d_K || !d_V || !d_O) return dh::fail(1, "[%s] null pointer", op);
  if ((reinterpret_cast<uintptr_t>(d_K) | reinterpret_cast<uintptr_t>(d_V) | reinterpret_cast<uintptr_t>(d_Q) |
       reinterpret_cast<uintptr_t>(d_O)) & 15)
    return dh::fail(1, "[%s] Q/K/V/O pointers must be 16-byte aligned", op);
  PrefillArgs a{};
  a.Q = d_Q; a.K = static_cast<const __half*>(d_K); a.V = static_cast<const __half*>(d_V); a.O = d_O;
  a.T = T; a.H = H; a.Hkv = Hkv; a.G = H / Hkv; a.kv_len = kv_len; a.start_pos = start_pos;
  a.causal = causal ? 1 : 0; a.window = sliding_window; a.scale = scale; a.softcap = softcap;
  // Two 16-query groups per wave halve the LDS traffic per product (H 32, T 2048: 73 -> 61 us, the fewest workgroups that gain);
  // short prompts keep 64-query tiles so that the grid still covers the compute units (H 16, T 2048: 37 us, 45 with 128).
  static const int env_qt = dh::tuning_int("DH_ATTN_PREFILL_QT", 0);
  const int qt = env_qt ? env_qt : ((int64_t)dh::ceil_div(T, 128) * H >= 2 * dh::num_cus() ? 2 : 1);
  const dim3 grid((unsigned)dh::ceil_div(T, 64 * qt), (unsigned)H);
  if (D == 64) {
    if (qt == 2) hipLaunchKernelGGL((attn_prefill_kernel<64, 64, 2, false>), grid, dim3(512), 0, dh::stream(), a);
    else hipLaunchKernelGGL((attn_prefill_kernel<64, 64, 1, false>), grid, dim3(512), 0, dh::stream(), a);
  } else {
    if (qt == 2) hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 2, false>), grid, dim3(512), 0, dh::stream(), a);
    else hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 1, false>), grid, dim3(512), 0, dh::stream(), a);
  }
  DH_CHECK_LAUNCH(op);
  return 0;
}

namespace {
template <int D, int VD>
int launch_spec(const char* op, const PrefillArgs& a) {
  static const int env_qt = dh::tuning_int("DH_ATTN_SPEC_QT", 0);
  // keys of more than 128 elements: two query groups would spill registers
  const int qt = D > 128 ? 1 : env_qt ? env_qt : dh::ceil_div(a.T, 128) * a.H >= 2 * dh::num_cus() ? 2 : 1;
  const dim3 grid((unsigned)dh::ceil_div(a.T, 64 * qt), (unsigned)a.H);
  if constexpr (D > 128) hipLaunchKernelGGL((attn_prefill_kernel<D, VD, 1, true>), grid, dim3(512), 0, dh::stream(), a);
  else if (qt == 2) hipLaunchKernelGGL((attn_prefill_kernel<D, VD, 2, true>), grid, dim3(512), 0, dh::stream(), a);
  else hipLaunchKernelGGL((attn_prefill_kernel<D, VD, 1, true>), grid, dim3(512), 0, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

// Prompts over f32 caches: attn_prefill_f32_kernel, or the general kernel where that is the faster of the two, which few queries over few
// key-value heads are (a workgroup of it is one query and up to eight heads of a key-value head, so its time goes with the heads at
// once; a workgroup here is 16 queries of one head).  Both take a start and a time for each key the last query sees, in us: the general
// kernel's by lanes a key (heads of at most 64 elements, of 128) and heads at once, and by how many workgroups a compute unit has; this
// one's by its instance and rounds of one workgroup on every compute unit.  Fitted to 4800 calls (heads of 32 .. 128, 4 .. 64 of them,
// 16 .. 200 queries, 16 .. 3200 keys) and checked on 1584 with windows of 16 .. 1024: the choice is 0.2 and 0.6 % behind the better of the
// two on average, at worst 1.2 us on 4.8.  General / this, H 8/8, D 128: 16 queries 4.4 / 8.3 us, 33 behind 500 keys 18 / 25, 200 21 / 13;
// H 16/8: 16 behind 3000 83 / 104, 100 behind 3000 209 / 104; H 32/8: 64 behind 500 38 / 27.  Fewer than 16 queries leave most of a tile
// empty.
bool takes_f32_tiles(const dh_attn_spec* s, int dk, int T, int start_pos) {
  if (dk > 128 || s->VD > 128 || T < 16 || s->H > 65535) return false;
  constexpr double general_start[2] = {5.1, 6.1};
  constexpr double general_key[2][4] = {{0.0084, 0.0147, 0.0231, 0.0398}, {0.0190, 0.0250, 0.0402, 0.0774}};
  constexpr double tiles_start[4] = {5.1, 6.4, 6.6, 6.8}, tiles_key[4] = {0.0141, 0.0228, 0.0239, 0.0313};
  const double cus = dh::num_cus(), keys = std::min<int64_t>((int64_t)start_pos + T, s->window > 0 ? s->window : INT32_MAX);
  const int G = s->H / s->Hkv, wide = dk > 64 || s->VD > 64, log2_heads = G <= 1 ? 0 : G <= 2 ? 1 : G <= 4 ? 2 : 3;
  const double per_cu = (double)s->Hkv * dh::ceil_div(G, 1 << log2_heads) * T / cus;
  const double general = general_start[wide] + keys * general_key[wide][log2_heads] * (per_cu <= 1.0 ? 1.0 : per_cu <= 2.0 ? 1.29 : 0.82 * per_cu);
  const int instance = 2 * (dk > 64) + (s->VD > 64);
  const int64_t rounds = dh::ceil_div(dh::ceil_div(T, 16) * s->H, dh::num_cus());
  return tiles_start[instance] + keys * tiles_key[instance] * rounds <= general;
}
}  // namespace

extern "C" int dh_attn_spec_prefill(const dh_attn_spec* spec, const float* d_qkv, const void* d_cache_k, const void* d_cache_v,
                                    void* d_out, int out_dtype, int ld_out, int T, int start_pos) {
  return dh_attn_spec_prefill_shared(spec, d_qkv, d_cache_k, nullptr, 0, 0, d_cache_v, d_out, out_dtype, ld_out, T, start_pos);
}

extern "C" int dh_attn_spec_prefill_shared(const dh_attn_spec* spec, const float* d_qkv, const void* d_cache_k, const void* d_shared_k,
                                           int shared_dim, int ld_shared, const void* d_cache_v, void* d_out, int out_dtype,
                                           int ld_out, int T, int start_pos) {
  const char* op = "dh_attn_spec_prefill";
  DH_REQUIRE_INIT(op);
  if (int rc = dh::attn_spec_check(op, spec)) return rc;
  if (T <= 0 || start_pos < 0) return dh::fail(1, "[%s] seqLen must be positive and startPos non-negative", op);
  if (out_dtype != DH_F32 && out_dtype != DH_BF16) return dh::fail(1, "[%s] output must be f32 or bf16, got dtype %d", op, out_dtype);
  if (ld_out < spec->H * spec->VD || ld_out % 4) return dh::fail(1, "[%s] ld_out=%d must be a multiple of 4 and hold %d elements", op, ld_out, spec->H * spec->VD);
  if (!d_qkv || !d_cache_k || !d_cache_v || !d_out) return dh::fail(1, "[%s] null pointer", op);
  if ((reinterpret_cast<uintptr_t>(d_qkv) | reinterpret_cast<uintptr_t>(d_cache_k) | reinterpret_cast<uintptr_t>(d_cache_v) |
       reinterpret_cast<uintptr_t>(d_out)) & 15)
    return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  const int dk = spec->D + shared_dim;
  if (shared_dim < 0 || shared_dim % 8 || dk > 512) return dh::fail(1, "[%s] %d shared key elements beside %d must be a multiple of 8, 512 in all", op, shared_dim, spec->D);
  if (shared_dim > 0 && (!d_shared_k || ld_shared < shared_dim || ld_shared % 8 || (reinterpret_cast<uintptr_t>(d_shared_k) & 15)))
    return dh::fail(1, "[%s] shared key rows must be 16-byte aligned and ld_shared=%d a multiple of 8 that holds %d elements", op, ld_shared, shared_dim);
  if (spec->ld_qkv < spec->H * dk) return dh::fail(1, "[%s] a projection row of %d floats does not hold its queries", op, spec->ld_qkv);
  const dh::SharedKey shared{d_shared_k, shared_dim, ld_shared};
  const bool wide_cache = spec->cache_dtype != DH_F16;
  if (wide_cache ? !takes_f32_tiles(spec, dk, T, start_pos) : dk > 256 || spec->VD > 128 || ld_shared >= 1 << 24)
    return dh::attn_spec_prefill_general(op, spec, d_qkv, d_cache_k, d_cache_v, d_out, out_dtype, ld_out, T, start_pos, shared);
  PrefillArgs a{};
  a.Q = d_qkv; a.K = static_cast<const __half*>(d_cache_k); a.V = static_cast<const __half*>(d_cache_v);
  a.O = out_dtype == DH_F32 ? static_cast<float*>(d_out) : nullptr;
  a.O16 = out_dtype == DH_BF16 ? static_cast<uint16_t*>(d_out) : nullptr;
  a.T = T; a.H = spec->H; a.Hkv = spec->Hkv; a.G = spec->H / spec->Hkv; a.kv_len = start_pos + T; a.start_pos = start_pos;
  a.causal = 1; a.window = spec->window; a.scale = spec->scale; a.softcap = 0.f;
  a.dk = dk; a.dv = spec->VD; a.own_k = spec->D; a.KS = static_cast<const __half*>(d_shared_k); a.ld_shared = ld_shared;
  a.ld_q = spec->ld_qkv; a.ld_o = ld_out;
  a.r1 = spec->d_bias_r1; a.r2 = spec->d_bias_r2;
  a.gate = spec->gate_offset >= 0 ? d_qkv + spec->gate_offset : nullptr;
  if (wide_cache) {
    const dim3 grid((unsigned)dh::ceil_div(T, 16), (unsigned)spec->H);
    if (dk <= 64 && spec->VD <= 64) hipLaunchKernelGGL((attn_prefill_f32_kernel<64, 64>), grid, dim3(512), 0, dh::stream(), a);
    else if (dk <= 64) hipLaunchKernelGGL((attn_prefill_f32_kernel<64, 128>), grid, dim3(512), 0, dh::stream(), a);
    else if (spec->VD <= 64) hipLaunchKernelGGL((attn_prefill_f32_kernel<128, 64>), grid, dim3(512), 0, dh::stream(), a);
    else hipLaunchKernelGGL((attn_prefill_f32_kernel<128, 128>), grid, dim3(512), 0, dh::stream(), a);
    DH_CHECK_LAUNCH(op);
    return 0;
  }
  if (dk <= 64) return spec->VD <= 64 ? launch_spec<64, 64>(op, a) : launch_spec<64, 128>(op, a);
  if (dk <= 128) return spec->VD <= 64 ? launch_spec<128, 64>(op, a) : launch_spec<128, 128>(op, a);
  return dk <= 192 ? launch_spec<192, 128>(op, a) : launch_spec<256, 128>(op, a);
}

extern "C" int dh_attn_spec_prefill_plan(const dh_attn_spec* spec, int shared_dim, int T, int start_pos, int num_cus) {
  const char* op = "dh_attn_spec_prefill_plan";
  if (dh::attn_spec_check(op, spec)) return -1;
  if (T <= 0 || start_pos < 0 || shared_dim < 0) {
    dh::fail(1, "[%s] seqLen must be positive, startPos and the shared elements non-negative", op);
    return -1;
  }
  const int dk = spec->D + shared_dim;
  if (spec->cache_dtype == DH_F16) return dk <= 256 && spec->VD <= 128 ? 1 : 0;
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  const bool tiles = takes_f32_tiles(spec, dk, T, start_pos);
  dh::plan_end();
  return tiles ? 1 : 0;
}
