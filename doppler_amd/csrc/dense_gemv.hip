// Products of ONE f32 activation row with dense bf16 weights (decode), HBM-bound.
//
// The row sits in LDS as f32 (optionally RMS-normalised on its way there); a wave streams one weight row at a time,
// 16 bytes per lane and load with the non-temporal hint, U loads of the next stage in flight while the current
// ones are multiplied (f32 fma on the widened weights, so the product is a 32-bit one).  The row (as far as a few pieces a thread hold it), its norm's
// weights, the first stage of weights and what an output adds and multiplies in are requested together: short products are a chain of trips to
// memory, and this makes them one.  (The weights' loads are conditional, so the compiler cannot count them, and the row is prepared when all of it has
// arrived, not while the weights travel.)  us, alone, weights from memory, against weights in front of a row that was requested when they had come: 2048 x 8192 with a
// residual 9.5 -> 8.9, 2048 x 1024 4.1 -> 3.7, 4096 x 4096 with a norm 8.7 -> 7.9, 3080 x 1024 4.6 -> 4.6, gated heads 1024 x 1024 4.8 -> 4.2, 32000 x 1024 18.7 -> 14.4.
// The row is kept as two planes of 16-byte pieces (elements 0..3 and 4..7 of every eight) so that a wave's reads of either plane are consecutive.
//
// Outputs as in the multi-row product (dense_gemm.hip): columns below n_first with bias, column scale and residual, the rest
// through an activation; or the argmax over all of them (output head).
//
// The ATTN form merges an attention's key splits (attention_spec.hip) into the front of the row: a launch less in front of the product.  A wave makes the
// factors of a few heads' splits (a lane each) from their maxima and weights, while the sums travel.
//
// The HEADS form reads the raw outputs of a layer's heads instead: each head divided by its root mean square, weighted and
// multiplied by the sigmoid of an output gate on its way into LDS.
#include <algorithm>
#include <cfloat>

#include "argmax_device.h"
#include "attention_spec.h"
#include "dense_device.h"

namespace {

using dh::Cand;

constexpr int kMaxK = 32768;
constexpr int kMaxHeads = 256;        // of the HEADS form

struct GemvArgs {
  const float* x;
  const float* norm_weight;   // null: the row as it is
  int hidden;                 // elements the norm's mean runs over
  float eps;
  const uint16_t* W;
  int64_t ldw;
  int N, K;
  float alpha;
  const float* bias;
  const float* residual;
  const float* col_scale;
  float* C;
  int n_first;
  float* C2;
  int act;
  const float* gate;          // HEADS form: one number per element; norm_weight has one too, eps is the heads'
  int heads, head_padded, head_size;
  const float* splits;        // ATTN form: [attn_heads][nsplit][attn_dim] sums, then as many pairs (maximum, weight); head_gate one number a head, or null
  const float* head_gate;
  int attn_heads, attn_dim, nsplit;
  dh::DynKeys keys;           // how many of the splits there are, where only the device knows
  int iters;                  // rows per wave
  float* part_val;            // argmax: per-workgroup candidates
  uint32_t* part_idx;
};

// What the row is made of.
enum RowForm { kPlainRow, kHeadsRow, kAttnRow };

template <int U, int WAVES, int BATCH, bool ARGMAX, int FORM>
__global__ __launch_bounds__(64 * WAVES) void gemv_kernel(const GemvArgs a) {
  extern __shared__ __align__(16) float4 planes[];      // [2][K / 8]
  __shared__ float red[WAVES];
  __shared__ float sv[WAVES];
  __shared__ uint32_t si[WAVES];
  constexpr int THREADS = 64 * WAVES;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int np = a.K >> 3, nstages = (np + 64 * U - 1) / (64 * U);
  const int units = a.iters * nstages;

  uint4 cur[U], nxt[U];
  struct Terms {               // of a row's output
    float bias, scale, residual;
  };
  Terms cur_terms, nxt_terms;
  auto row_of = [&](int it) { return (int64_t)(it * (int)gridDim.x + (int)blockIdx.x) * WAVES + wave; };
  auto load = [&](int unit, uint4 (&dst)[U], Terms& terms) {
    const int it = unit / nstages, st = unit - it * nstages;
    const uint4* w = reinterpret_cast<const uint4*>(a.W + min(row_of(it), (int64_t)a.N - 1) * a.ldw);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int p = lane + 64 * (u + U * st);
      dst[u] = p < np ? dh::stream_load_16(w + p) : make_uint4(0, 0, 0, 0);
    }
    if (!ARGMAX && st == 0) {
      const int64_t n = min(row_of(it), (int64_t)a.n_first - 1);
      terms = Terms{0.f, 1.f, 0.f};
      if (n >= 0) {
        if (a.bias) terms.bias = a.bias[n];
        if (a.col_scale) terms.scale = a.col_scale[n];
        if (a.residual) terms.residual = a.residual[n];
      }
    }
  };

  // ---- the activation row
  if constexpr (FORM == kAttnRow) {
    constexpr int HB = 4, SB = 8;                        // heads a wave, splits a piece that are requested at once
    extern __shared__ __align__(16) float4 planes_and_factors[];
    float* const factors = reinterpret_cast<float*>(planes_and_factors) + a.K;      // [heads][nsplit]
    float* const inverse = factors + a.attn_heads * a.nsplit;                       // [heads]
    const int vp = a.attn_dim >> 2, live = a.attn_heads * vp, pieces = a.K >> 2, stride = a.nsplit;
    const float4 *sums = reinterpret_cast<const float4*>(a.splits), *xg = reinterpret_cast<const float4*>(a.x);
    const float2* pairs = reinterpret_cast<const float2*>(a.splits + (int64_t)a.attn_heads * stride * a.attn_dim);
    const int nsplit = a.keys.kv_len_ptr ? dh::dyn_key_range(a.keys).nsplit : stride;
    // a thread's first piece of the heads' part (its first splits) and of the rest, a wave's first heads, the first weights
    float2 pair[HB];
    float gate[HB];
    auto head_of = [&](int j) { return min(wave + WAVES * j, a.attn_heads - 1); };
    auto pair_of = [&](int h) { return pairs[h * stride + max(min(lane, nsplit - 1), 0)]; };
#pragma unroll
    for (int j = 0; j < HB; j++) {
      pair[j] = pair_of(head_of(j));
      gate[j] = a.head_gate ? a.head_gate[head_of(j)] : 0.f;
    }
    float4 part[SB], rest[BATCH];
    auto part_of = [&](int i, int s) { return sums[((i / vp) * stride + max(min(s, nsplit - 1), 0)) * vp + i % vp]; };
    const int turned = (int)((tid + 64 * blockIdx.x) % THREADS);         // workgroups begin at different heads: they read the same lines
#pragma unroll
    for (int s = 0; s < SB; s++) part[s] = part_of(min(turned, live - 1), s);
#pragma unroll
    for (int b = 0; b < BATCH; b++) rest[b] = xg[min(live + tid + THREADS * b, pieces - 1)];
    load(0, cur, cur_terms);
    auto make_factors = [&](int h, const float2& p, float g) {
      const bool there = lane < nsplit;
      const float M = dh::group_combine<1, 64>(there ? p.x : -FLT_MAX, dh::MaxOp());
      const float f = there ? __builtin_amdgcn_exp2f(p.x - M) : 0.f;
      const float den = dh::wave_sum_uniform(there ? fmaf(f, p.y, 0.f) : 0.f);
      if (there) factors[h * stride + lane] = f;
      if (lane == 0) inverse[h] = (den > 0.f ? 1.0f / den : 0.f) * (a.head_gate ? 1.0f / (1.0f + expf(-g)) : 1.0f);
    };
#pragma unroll
    for (int j = 0; j < HB; j++)
      if (wave + WAVES * j < a.attn_heads) make_factors(wave + WAVES * j, pair[j], gate[j]);
    for (int h = wave + WAVES * HB; h < a.attn_heads; h += WAVES) make_factors(h, pair_of(h), a.head_gate ? a.head_gate[h] : 0.f);
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int i = live + tid + THREADS * b;
      if (i < pieces) planes[(i & 1) * np + (i >> 1)] = rest[b];
    }
    for (int i = live + tid + THREADS * BATCH; i < pieces; i += THREADS) planes[(i & 1) * np + (i >> 1)] = xg[i];
    __syncthreads();
    for (int i = turned; i < live; i += THREADS) {
      const int h = i / vp;
      float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int s0 = 0; s0 < nsplit; s0 += SB) {
        if (i != turned || s0 > 0) {
#pragma unroll
          for (int s = 0; s < SB; s++) part[s] = part_of(i, s0 + s);
        }
#pragma unroll
        for (int s = 0; s < SB; s++) {
          if (s0 + s >= nsplit) break;
          const float f = factors[h * stride + s0 + s];
          y.x = fmaf(f, part[s].x, y.x); y.y = fmaf(f, part[s].y, y.y); y.z = fmaf(f, part[s].z, y.z); y.w = fmaf(f, part[s].w, y.w);
        }
      }
      const float inv = inverse[h];
      planes[(i & 1) * np + (i >> 1)] = make_float4(y.x * inv, y.y * inv, y.z * inv, y.w * inv);
    }
  } else if constexpr (FORM == kHeadsRow) {
    // weighted and gated on the way in; the squares are summed by eight lanes (whole heads: their sizes are multiples of 32), then by
    // head, and the row in LDS is scaled last: one trip to memory
    __shared__ float inv_s[kMaxHeads];
    __shared__ float squares[kMaxK / 32];
    const int hp = a.head_padded >> 2, live = a.heads * hp;       // 16-byte pieces of a head, of all heads
    auto piece_of = [&](const float* row, int i) {
      const float4 x = reinterpret_cast<const float4*>(row)[min(i, live - 1)];
      return i < live ? x : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    auto put = [&](int i, float4 y, const float4& w, const float4& g) {
      float ss = fmaf(y.x, y.x, fmaf(y.y, y.y, fmaf(y.z, y.z, y.w * y.w)));
      y.x = y.x * w.x * __frcp_rn(1.0f + __expf(-g.x)); y.y = y.y * w.y * __frcp_rn(1.0f + __expf(-g.y));
      y.z = y.z * w.z * __frcp_rn(1.0f + __expf(-g.z)); y.w = y.w * w.w * __frcp_rn(1.0f + __expf(-g.w));
      planes[(i & 1) * np + (i >> 1)] = y;
      ss = dh::group_combine<1, 8>(ss, dh::AddOp());
      if ((i & 7) == 0) squares[i >> 3] = ss;
    };
    float4 v[BATCH], w[BATCH], g[BATCH];
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int i = tid + THREADS * b;
      v[b] = piece_of(a.x, i); w[b] = piece_of(a.norm_weight, i); g[b] = piece_of(a.gate, i);
    }
    load(0, cur, cur_terms);
#pragma unroll
    for (int b = 0; b < BATCH; b++)
      if (tid + THREADS * b < (a.K >> 2)) put(tid + THREADS * b, v[b], w[b], g[b]);      // sixteen lanes at a time: K is a multiple of 64
    for (int i = tid + THREADS * BATCH; i < (a.K >> 2); i += THREADS) put(i, piece_of(a.x, i), piece_of(a.norm_weight, i), piece_of(a.gate, i));
    __syncthreads();
    for (int h = tid; h < a.heads; h += THREADS) {
      float ss = 0.f;
      for (int k = h * (hp >> 3); k < (h + 1) * (hp >> 3); k++) ss += squares[k];
      inv_s[h] = 1.0f / sqrtf(ss / (float)a.head_size + a.eps);
    }
    __syncthreads();
    for (int i = tid; i < live; i += THREADS) {
      const float f = inv_s[i / hp];
      float4& v = planes[(i & 1) * np + (i >> 1)];
      v.x *= f; v.y *= f; v.z *= f; v.w *= f;
    }
  } else {
    const float4 *xg = reinterpret_cast<const float4*>(a.x), *wg = reinterpret_cast<const float4*>(a.norm_weight);
    const int pieces = a.K >> 2;
    float4 v[BATCH], w[BATCH];
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int i = min(tid + THREADS * b, pieces - 1);
      v[b] = xg[i];
      w[b] = wg ? wg[i] : make_float4(1.f, 1.f, 1.f, 1.f);
    }
    load(0, cur, cur_terms);
    float inv = 1.f;
    if (wg) {
      float ss = 0.f;
      auto square = [&](const float4& p) {
        ss = fmaf(p.x, p.x, ss); ss = fmaf(p.y, p.y, ss); ss = fmaf(p.z, p.z, ss); ss = fmaf(p.w, p.w, ss);
      };
#pragma unroll
      for (int b = 0; b < BATCH; b++)
        if (tid + THREADS * b < pieces) square(v[b]);
      for (int i = tid + THREADS * BATCH; i < pieces; i += THREADS) square(xg[i]);
      ss = dh::wave_sum_uniform(ss);
      if (lane == 0) red[wave] = ss;
      __syncthreads();
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; w++) total += red[w];
      inv = 1.0f / sqrtf(total / (float)a.hidden + a.eps);
    }
    auto put = [&](int i, float4 y, const float4& f) {
      if (wg) y = make_float4(y.x * inv * f.x, y.y * inv * f.y, y.z * inv * f.z, y.w * inv * f.w);
      planes[(i & 1) * np + (i >> 1)] = y;
    };
#pragma unroll
    for (int b = 0; b < BATCH; b++)
      if (tid + THREADS * b < pieces) put(tid + THREADS * b, v[b], w[b]);
#pragma unroll 2
    for (int i = tid + THREADS * BATCH; i < pieces; i += THREADS) put(i, xg[i], wg ? wg[i] : make_float4(1.f, 1.f, 1.f, 1.f));
  }
  __syncthreads();

  float acc = 0.f;
  Cand best{-FLT_MAX, 0xFFFFFFFFu};
  int st = 0, it = 0;
  for (int unit = 0; unit < units; unit++) {
    nxt_terms = cur_terms;
    if (unit + 1 < units) load(unit + 1, nxt, nxt_terms);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int p = min(lane + 64 * (u + U * st), np - 1);      // past the row the weights are zeros
      const float4 xa = planes[p], xb = planes[np + p];
      const uint4 w = cur[u];
      acc = fmaf(xa.x, dh::bf16_low(w.x), acc); acc = fmaf(xa.y, dh::bf16_high(w.x), acc);
      acc = fmaf(xa.z, dh::bf16_low(w.y), acc); acc = fmaf(xa.w, dh::bf16_high(w.y), acc);
      acc = fmaf(xb.x, dh::bf16_low(w.z), acc); acc = fmaf(xb.y, dh::bf16_high(w.z), acc);
      acc = fmaf(xb.z, dh::bf16_low(w.w), acc); acc = fmaf(xb.w, dh::bf16_high(w.w), acc);
    }
    if (++st == nstages) {
      const float v = dh::wave_sum_uniform(acc) * a.alpha;
      acc = 0.f;
      const int64_t n = row_of(it);
      if (lane == 0 && n < a.N) {
        if (n < a.n_first) {
          float y = v;
          if constexpr (!ARGMAX) {
            y += cur_terms.bias;
            if (a.col_scale) y *= cur_terms.scale;
            if (a.residual) y += cur_terms.residual;
          }
          if (a.C) a.C[n] = y;
        } else {
          a.C2[n - a.n_first] = dh::activate(v, a.act);
        }
        if (ARGMAX && dh::beats(v, (uint32_t)n, best.v, best.i)) { best.v = v; best.i = (uint32_t)n; }
      }
      st = 0;
      it++;
    }
#pragma unroll
    for (int u = 0; u < U; u++) cur[u] = nxt[u];
    cur_terms = nxt_terms;
  }
  if (ARGMAX) {
    if (lane == 0) { sv[wave] = best.v; si[wave] = best.i; }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < WAVES; w++)
        if (dh::beats(sv[w], si[w], best.v, best.i)) { best.v = sv[w]; best.i = si[w]; }
      a.part_val[blockIdx.x] = best.v;
      a.part_idx[blockIdx.x] = best.i;
    }
  }
}

// BATCH: 16-byte pieces of the row that a thread requests in front of the weights.
template <int U, int WAVES, int BATCH, bool ARGMAX, int FORM>
int launch(const char* op, GemvArgs a, int max_grid, int* parts) {
  auto kern = gemv_kernel<U, WAVES, BATCH, ARGMAX, FORM>;
  static bool attr_set = false;
  if (!attr_set) {
    DH_CHECK_HIP(op, hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         kMaxK * 4 + (FORM == kAttnRow ? dh::kMergedFactors : 0)));
    attr_set = true;
  }
  if (ARGMAX) max_grid = std::min(max_grid, dh::kMaxParts);
  const int64_t groups = dh::ceil_div(a.N, WAVES);
  a.iters = (int)std::max<int64_t>(1, dh::ceil_div(groups, max_grid));
  const int grid = (int)dh::ceil_div(groups, a.iters);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WAVES), (size_t)a.K * 4 + (FORM == kAttnRow ? (size_t)4 * a.attn_heads * (a.nsplit + 1) : 0),
                     dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  if (parts) *parts = grid;
  return 0;
}

template <int WAVES, bool ARGMAX, int FORM>
int launch_loads(const char* op, const GemvArgs& a, int max_grid, int* parts) {
  // a stage as long as the row: lanes past the end load nothing and multiply zeros (a row of 1024 in a stage of 4096 leaves a quarter
  // of the bytes in flight).  Four waves a workgroup are few, so long rows get long stages there, and gated heads where a row is all a wave
  // has (2048 x 4096 7.5 -> 7.1 us) or very long (4096 x 8192 19.3 -> 16.9); two stages of 1536 fit rows up to 3072 better than two of
  // 2048 (2560 x 2560 5.9 -> 5.5).
  // Pieces: what a row up to the stage's length has for a thread.  Requests for more of them stand in front of the weights for nothing (us, two or
  // four pieces / one: norm 1536 x 1024 4.2 -> 3.9, 3080 x 1024 4.8 -> 4.6, 2050 x 2048 5.1 -> 4.9, heads 1024 x 1024 4.4 -> 4.2); output heads, with
  // many rows a wave, go better with two (32000 x 2048 21.1 against 22.0).  Longer rows: as many as registers allow (four workgroups of eight waves: 64).
  constexpr bool HEADS = FORM == kHeadsRow;
  constexpr int BATCH = HEADS || WAVES == 4 ? 4 : 2;
  if (a.K <= 1024) return launch<2, WAVES, ARGMAX ? 2 : 1, ARGMAX, FORM>(op, a, max_grid, parts);
  if (a.K <= 2048) return launch<4, WAVES, ARGMAX || WAVES == 4 ? 2 : 1, ARGMAX, FORM>(op, a, max_grid, parts);
  if constexpr (WAVES == 4) return launch<8, WAVES, BATCH, ARGMAX, FORM>(op, a, max_grid, parts);
  if constexpr (HEADS) {
    if (WAVES == 8 ? a.N <= 8 * dh::num_cus() : a.K > 4096) return launch<8, WAVES, BATCH, ARGMAX, FORM>(op, a, max_grid, parts);
  } else {
    if (a.K <= 3072) return launch<3, WAVES, BATCH, ARGMAX, FORM>(op, a, max_grid, parts);
  }
  return launch<4, WAVES, BATCH, ARGMAX, FORM>(op, a, max_grid, parts);
}

// Rows of each of its workgroups that the busiest compute unit goes through, with at most `per_cu` workgroups on every one.
int64_t busiest(int64_t N, int waves, int per_cu) {
  const int64_t cus = dh::num_cus(), groups = dh::ceil_div(N, waves), iters = dh::ceil_div(groups, per_cu * cus);
  return dh::ceil_div(dh::ceil_div(groups, iters), cus) * iters;
}

// Every workgroup prepares the whole activation row, so workgroups are as wide as leaves one for every compute unit, and as many
// as are resident at once; of rows beyond 2048 two to a compute unit, or four where that spreads them better (5136 rows are 642 groups:
// two rounds of 321, or one of 642; x 2560 8.9 -> 6.9 us, x 8192 17.4 -> 16.7).  us, N x K with four waves and stages of 4096 (or two rows of 2048) -> now,
// weights from memory: 10256 x 2048 10.6 -> 9.8, 5136 x 1024 5.9 -> 4.5, 18464 x 4096 28.0 -> 25.8 (5.9 TB/s), 2050 x 8192 9.8 -> 9.1; with
// a norm 5136 x 1024 6.3 -> 5.1, 5136 x 2048 8.1 -> 7.1; heads 32000 x 2048 27.1 -> 25.6, 32000 x 1024 18.6 -> 16.9.  A launch alone is about 4 of them.
template <bool ARGMAX, int FORM = kPlainRow>
int dispatch(const char* op, const GemvArgs& a, int* parts) {
  constexpr bool HEADS = FORM == kHeadsRow;
  const int cus = dh::num_cus();
  if (a.K > 8192) return launch<8, 8, HEADS ? 4 : 2, ARGMAX, FORM>(op, a, a.K <= 16384 ? 2 * cus : cus, parts);
  if constexpr (HEADS)          // three rows are read to prepare one
    if (a.N >= 16 * cus) return launch_loads<16, ARGMAX, FORM>(op, a, cus, parts);
  if (a.N >= 8 * cus) {
    const bool four = !HEADS && (a.K <= 2048 || busiest(a.N, 8, 4) < busiest(a.N, 8, 2));
    return launch_loads<8, ARGMAX, FORM>(op, a, four ? 4 * cus : 2 * cus, parts);
  }
  return launch_loads<4, ARGMAX, FORM>(op, a, 4 * cus, parts);
}

int check(const char* op, const float* x, const float* norm_weight, int hidden, float eps, const void* W, int ldw, int N, int K) {
  if (N <= 0 || K <= 0) return dh::fail(1, "[%s] Dimensions must be positive: N=%d, K=%d", op, N, K);
  if (K % 64 || K > kMaxK) return dh::fail(1, "[%s] K=%d must be a multiple of 64 and at most %d", op, K, kMaxK);
  if (ldw < K || ldw % 8) return dh::fail(1, "[%s] ldw=%d must be a multiple of 8 and hold K=%d elements", op, ldw, K);
  if (!x || !W) return dh::fail(1, "[%s] null pointer", op);
  if (norm_weight && (hidden <= 0 || hidden > K || !(eps >= 0.f)))
    return dh::fail(1, "[%s] the norm needs 0 < hidden <= K and eps >= 0 (hidden=%d, K=%d)", op, hidden, K);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(norm_weight)) & 15)
    return dh::fail(1, "[%s] activation, norm and weight pointers must be 16-byte aligned", op);
  return 0;
}

GemvArgs make_args(const float* x, const float* norm_weight, int hidden, float eps, const void* W, int ldw, int N, int K,
                   float alpha) {
  GemvArgs a{};
  a.x = x; a.norm_weight = norm_weight; a.hidden = hidden; a.eps = eps;
  a.W = static_cast<const uint16_t*>(W); a.ldw = ldw; a.N = N; a.K = K; a.alpha = alpha; a.n_first = N;
  a.act = DH_ACT_NONE;
  return a;
}

}  // namespace

extern "C" {

int dh_dense_gemv(const float* d_x, const float* d_norm_weight, int hidden, float eps, const void* d_W, int ldw, int N,
                  int K, float alpha, const float* d_bias, const float* d_residual, float* d_C, int n_first, float* d_C2,
                  int activation) {
  return dh_dense_gemv_scaled(d_x, d_norm_weight, hidden, eps, d_W, ldw, N, K, alpha, d_bias, nullptr, d_residual, d_C, n_first, d_C2,
                              activation);
}

int dh_dense_gemv_scaled(const float* d_x, const float* d_norm_weight, int hidden, float eps, const void* d_W, int ldw, int N,
                         int K, float alpha, const float* d_bias, const float* d_col_scale, const float* d_residual, float* d_C,
                         int n_first, float* d_C2, int activation) {
  const char* op = "dh_dense_gemv";
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, d_x, d_norm_weight, hidden, eps, d_W, ldw, N, K)) return rc;
  if (n_first < 0 || n_first > N) return dh::fail(1, "[%s] n_first=%d is outside 0..%d", op, n_first, N);
  if ((n_first > 0 && !d_C) || (n_first < N && !d_C2)) return dh::fail(1, "[%s] null output pointer", op);
  if (d_x == d_C || d_x == d_C2) return dh::fail(1, "[%s] an output must not be the activation row", op);
  GemvArgs a = make_args(d_x, d_norm_weight, hidden, eps, d_W, ldw, N, K, alpha);
  a.bias = d_bias; a.col_scale = d_col_scale; a.residual = d_residual; a.C = d_C; a.n_first = n_first; a.C2 = d_C2; a.act = activation;
  return dispatch<false>(op, a, nullptr);
}

int dh_dense_gemv_heads(const float* d_x, const float* d_gate, const float* d_weight, int H, int padded, int size, float eps, const void* d_W,
                        int ldw, int N, int K, const float* d_col_scale, const float* d_residual, float* d_C) {
  const char* op = "dh_dense_gemv_heads";
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, d_x, nullptr, 0, eps, d_W, ldw, N, K)) return rc;
  if (H <= 0 || H > kMaxHeads || size <= 0 || padded < size || padded % 32 || (int64_t)H * padded > K)
    return dh::fail(1, "[%s] %d heads (at most %d) of %d elements, %d apart (a multiple of 32), in a row of %d", op, H, kMaxHeads, size, padded, K);
  if (!d_gate || !d_weight || !d_C) return dh::fail(1, "[%s] null pointer", op);
  if ((reinterpret_cast<uintptr_t>(d_gate) | reinterpret_cast<uintptr_t>(d_weight)) & 15) return dh::fail(1, "[%s] gate and weight must be 16-byte aligned", op);
  if (d_x == d_C) return dh::fail(1, "[%s] the output must not be the activation row", op);
  GemvArgs a = make_args(d_x, d_weight, 0, eps, d_W, ldw, N, K, 1.f);
  a.gate = d_gate; a.heads = H; a.head_padded = padded; a.head_size = size;
  a.col_scale = d_col_scale; a.residual = d_residual; a.C = d_C;
  return dispatch<false, kHeadsRow>(op, a, nullptr);
}

int dh_dense_gemv_attn(const dh_attn_spec* spec, const float* d_qkv, const void* d_workspace, int left, const uint32_t* d_kv_len, int max_kv_len,
                       const float* d_x, const void* d_W, int ldw, int N, int K, const float* d_residual, float* d_C) {
  const char* op = "dh_dense_gemv_attn";
  DH_REQUIRE_INIT(op);
  if (int rc = dh::attn_spec_check(op, spec)) return rc;
  if (int rc = check(op, d_x, nullptr, 0, 0.f, d_W, ldw, N, K)) return rc;
  if ((int64_t)spec->H * spec->VD > K || left <= 0 || !dh::product_merges(spec->H, left))
    return dh::fail(1, "[%s] %d splits of %d heads of %d elements in a row of %d", op, left, spec->H, spec->VD, K);
  if (!d_qkv || !d_workspace || !d_C) return dh::fail(1, "[%s] null pointer", op);
  if (reinterpret_cast<uintptr_t>(d_workspace) & 15) return dh::fail(1, "[%s] the workspace must be 16-byte aligned", op);
  if (d_kv_len && max_kv_len <= 0) return dh::fail(1, "[%s] max_kv_len must be positive with the key count on the device", op);
  // (the device's count decides how many are read, up to this many)
  if (d_kv_len && left != dh::attn_spec_wide_splits(spec, max_kv_len))
    return dh::fail(1, "[%s] %d splits are not those of up to %d keys", op, left, max_kv_len);
  if (d_x == d_C) return dh::fail(1, "[%s] the output must not be the activation row", op);
  GemvArgs a = make_args(d_x, nullptr, 0, 0.f, d_W, ldw, N, K, 1.f);
  a.residual = d_residual; a.C = d_C;
  a.splits = static_cast<const float*>(d_workspace); a.head_gate = spec->gate_offset >= 0 ? d_qkv + spec->gate_offset : nullptr;
  a.attn_heads = spec->H; a.attn_dim = spec->VD; a.nsplit = left;
  if (d_kv_len) a.keys = dh::attn_spec_keys(spec, d_kv_len, max_kv_len, true);
  return dispatch<false, kAttnRow>(op, a, nullptr);
}

static int lmhead_argmax(const char* op, const float* d_x, const float* d_norm_weight, int hidden, float eps, const void* d_W, int ldw,
                         int vocab, int K, float alpha, void* d_workspace, uint32_t* d_token_out, int output_index,
                         float* d_logits_out, uint32_t* also) {
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, d_x, d_norm_weight, hidden, eps, d_W, ldw, vocab, K)) return rc;
  if (!d_workspace || !d_token_out) return dh::fail(1, "[%s] null pointer", op);
  if (output_index < 0) return dh::fail(1, "[%s] outputIndex must be non-negative", op);
  GemvArgs a = make_args(d_x, d_norm_weight, hidden, eps, d_W, ldw, vocab, K, alpha);
  a.C = d_logits_out;
  a.part_val = static_cast<float*>(d_workspace);
  a.part_idx = reinterpret_cast<uint32_t*>(static_cast<char*>(d_workspace) + (size_t)dh::kMaxParts * 4);
  int parts = 0;
  if (int rc = dispatch<true>(op, a, &parts)) return rc;
  return dh::launch_argmax_final(op, a.part_val, a.part_idx, parts, d_token_out, output_index, also);
}

int dh_dense_lmhead_argmax(const float* d_x, const float* d_norm_weight, int hidden, float eps, const void* d_W, int ldw,
                           int vocab, int K, float alpha, void* d_workspace, uint32_t* d_token_out, int output_index,
                           float* d_logits_out) {
  return lmhead_argmax("dh_dense_lmhead_argmax", d_x, d_norm_weight, hidden, eps, d_W, ldw, vocab, K, alpha, d_workspace, d_token_out, output_index,
                       d_logits_out, nullptr);
}

int dh_dense_lmhead_argmax_read(const float* d_x, const float* d_norm_weight, int hidden, float eps, const void* d_W, int ldw,
                                int vocab, int K, float alpha, void* d_workspace, uint32_t* d_token_out, int output_index,
                                float* d_logits_out, uint32_t* host_token) {
  const char* op = "dh_dense_lmhead_argmax_read";
  DH_REQUIRE_INIT(op);
  if (!host_token) return dh::fail(1, "[%s] no place for the token", op);
  return dh::read_with(op, host_token, 1, [&](uint32_t* also) {
    return lmhead_argmax(op, d_x, d_norm_weight, hidden, eps, d_W, ldw, vocab, K, alpha, d_workspace, d_token_out, output_index, d_logits_out, also);
  });
}

}  // extern "C"
