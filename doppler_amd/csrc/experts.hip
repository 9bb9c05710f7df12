// Mixtures of experts (dh_experts): every token uses the `top` experts with the largest router logits z, each weighted with
// sigmoid(z), and a shared expert weighted with sigmoid of one more logit.
//
//   expert(x) = W_down glu(W_gate x, W_up x),   glu(g, u) = g' sigmoid(1.702 g') (clamp(u, +-limit) + 1),  g' = min(g, limit)
//   out       = sum over chosen e of expert_e(s_e h) + sigmoid(z_shared) expert_shared(h)
//
// A weight multiplies its expert's input, so it scales the gate and up products in front of the clamps; the products
// themselves always read h.  The shared expert's weight scales its activations.
//
// Gate and up rows alternate in blocks of 32 (the matrix-core epilogue wants both of a column in one lane).
//
// Decode: experts_up_kernel chooses the experts itself (every workgroup, from the few logits), norms the row and streams the
// chosen gate and up rows; experts_down_kernel streams the chosen down matrices and the shared one side by side along k.
// Prefill: experts_router_kernel (logits and choices) and experts_place_kernel (rows sorted by expert, table of row tiles), or for f32 operands, many
// logits, long rows and long portions (routes_itself) a product, experts_route_kernel and experts_sort_kernel; grouped products on the matrix cores (dense_gemm.hip);
// experts_combine_kernel.
#include <algorithm>
#include <cfloat>

#include "argmax_device.h"
#include "experts.h"

namespace {

constexpr int kMaxTop = 32;
constexpr int kMaxExperts = 1024;

struct StepArgs {
  const float* x;
  const float* norm;
  const uint16_t* router;  // [E and the shared expert's][K]
  float* z;                // router logits [E], then the shared expert's
  const uint16_t* up;      // [E][2 ff][ld_in]
  const uint16_t* down;    // [E][hidden][ff]
  const uint16_t* shared_up;
  const uint16_t* shared_down;
  const float* ls;         // [hidden] or null
  float* act;              // [top ff + shared_ff]
  float* out;              // residual row, added to
  int hidden, K, E, top, ff, shared_ff;
  float eps, limit, shared_limit;
};

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }

// The top experts of a row of logits, by one wave: ids (and logits) in the order of their size, the lower id first among equals.
// Lane l holds experts l, l + 64, .., 64 SLOTS in all; the maximum is found by lane steps, its lowest holder from a ballot.
template <int SLOTS>
__device__ __forceinline__ void choose_upto(const float* z, int E, int top, int* ids, float* zs) {
  const int lane = threadIdx.x & 63;
  float v[SLOTS];
#pragma unroll
  for (int j = 0; j < SLOTS; j++) v[j] = lane + 64 * j < E ? z[lane + 64 * j] : -INFINITY;
  for (int t = 0; t < top; t++) {
    float best = v[0];
#pragma unroll
    for (int j = 1; j < SLOTS; j++) best = fmaxf(best, v[j]);
    const float mx = dh::group_combine<1, 64>(best, dh::MaxOp());
    int id = 0;                                          // logits that are not numbers: some expert, inside the tables
    bool found = false;
#pragma unroll
    for (int j = 0; j < SLOTS; j++) {
      const unsigned long long at = __builtin_amdgcn_ballot_w64(v[j] == mx && lane + 64 * j < E);
      if (!found && at != 0) {
        id = 64 * j + __builtin_ctzll(at);
        found = true;
      }
    }
    if (lane == 0) {
      ids[t] = id;
      zs[t] = mx;
    }
#pragma unroll
    for (int j = 0; j < SLOTS; j++)
      if (lane + 64 * j == id) v[j] = -INFINITY;
  }
}
// The same for up to 64 experts, a lane each: a lane's place is the number of experts in front of it.  The largest one after the other are `top` chains of
// lane steps (0.3 us each), this a pass over the experts whose steps do not wait for one another: experts_up and _down at hidden 1024, four of 16 experts,
// 6.6 against 6.9 and 4.8 against 5.0 us.  It costs by the experts and the other by the choices: a portion of eight tokens, us, the largest one after the other /
// this, 8 of 8 experts 25.6 / 24.7, 3 of 16 23.3 / 23.3, 2 of 16 23.2 / 23.3, 6 of 32 24.7 / 24.7, 2 of 32 23.2 / 23.8, 8 of 48 25.6 / 25.7, 8 of 64 25.4 / 25.8,
// 2 of 64 22.7 / 24.0.
__device__ __forceinline__ void choose_by_places(const float* z, int E, int top, int* ids, float* zs) {
  const int lane = threadIdx.x & 63;
  const float own = z[min(lane, E - 1)], key = lane < E && own == own ? own : -INFINITY;
  int place = 0;
  for (int j0 = 0; j0 < E; j0 += 8) {                  // (lanes past the last expert are in front of none)
#pragma unroll
    for (int j = j0; j < j0 + 8; j++) {
      const float other = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(key), j));
      place += other > key || (other == key && j < lane) ? 1 : 0;
    }
  }
  if (lane < E && place < top) {
    ids[place] = lane;
    zs[place] = own;
  }
  if (__builtin_popcountll(__builtin_amdgcn_ballot_w64(key > -INFINITY)) < top) {
    // choices behind the last logit above -infinity: the first number's expert again, for nothing (as above, where no number of 64 leaves the first as it is)
    const unsigned long long numbers = __builtin_amdgcn_ballot_w64(lane < E && own == own);
    if (lane < E && place < top && key == -INFINITY) {
      ids[place] = numbers ? __builtin_ctzll(numbers) : 0;
      if (numbers != 0 || E < 64 || place > 0) zs[place] = -INFINITY;
    }
  }
}
__device__ __forceinline__ void choose(const float* z, int E, int top, int* ids, float* zs) {
  if (E <= 64 && E <= 5 * top) choose_by_places(z, E, top, ids, zs);
  else if (E <= 64) choose_upto<1>(z, E, top, ids, zs);
  else if (E <= 256) choose_upto<4>(z, E, top, ids, zs);
  else choose_upto<kMaxExperts / 64>(z, E, top, ids, zs);
}

// A wave takes a gate and an up row at a time; the row sits in LDS as two planes of 16-byte pieces, as in the dense GEMV.
//
// PR > 0: the router's logits are made here too, by every workgroup, four waves five rows each of at most 64 PR pieces, requested beside the row itself;
// the first workgroup leaves them for experts_down_kernel.  A launch for seventeen sums (2.9 us and 1.4 in front of the next) against their weights once
// more for each workgroup, from the L2: us, 17 rows of 1024 7.8 against 2.8 + 6.6, of 2048 14.8 against 3.4 + 14.2, and a gap between
// launches less; from 4096 on the workgroups of a compute unit would read half a megabyte of them.  A wave whose first columns are the shared expert's requests those at once as well.
constexpr int kRouterRows = 5;                         // of a wave
template <int U, int PR>
__global__ __launch_bounds__(256) void experts_up_kernel(const StepArgs a, int iters) {
  extern __shared__ __align__(16) float4 planes[];       // [2][K / 8]
  __shared__ float red[4];
  __shared__ float logits_s[4 * kRouterRows];
  __shared__ int ids[kMaxTop];
  __shared__ float zs[kMaxTop];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int np = a.K >> 3, nstages = (np + 64 * U - 1) / (64 * U), total = a.top * a.ff + a.shared_ff;
  uint4 cur[2][U], nxt[2][U];
  auto load = [&](int unit, uint4 (&dst)[2][U]) {
    const int it = unit / nstages, st = unit - it * nstages;
    const int col = min((it * (int)gridDim.x + (int)blockIdx.x) * 4 + wave, total - 1);
    const bool shared = col >= a.top * a.ff;
    const int c = shared ? col - a.top * a.ff : col % a.ff;
    const uint16_t* m = shared ? a.shared_up : a.up + (int64_t)ids[col / a.ff] * 2 * a.ff * a.K;
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const uint4* w = reinterpret_cast<const uint4*>(m + (int64_t)(64 * (c >> 5) + 32 * r + (c & 31)) * a.K);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int p = lane + 64 * (u + U * st);
        dst[r][u] = p < np ? dh::stream_load_16(w + p) : make_uint4(0, 0, 0, 0);
      }
    }
  };
  const float4 *xg = reinterpret_cast<const float4*>(a.x), *wg = reinterpret_cast<const float4*>(a.norm);
  auto scaled = [](const float4& v, float f, const float4& w) { return make_float4(v.x * f * w.x, v.y * f * w.y, v.z * f * w.z, v.w * f * w.w); };
  auto squares = [](const float4& v, float ss) {
    ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss);
    return fmaf(v.w, v.w, ss);
  };
  const float* z = a.z;
  if constexpr (PR > 0) {
    constexpr int XV = (PR + 1) / 2;                     // pieces of the row a thread holds
    const int rows = a.E + (a.shared_ff ? 1 : 0), nx = a.K >> 2;
    const bool ahead = (int)blockIdx.x * 4 >= a.top * a.ff;
    float4 xv[XV], wv[XV];
    uint4 rw[kRouterRows][PR];
#pragma unroll
    for (int j = 0; j < XV; j++) {
      xv[j] = xg[min(tid + 256 * j, nx - 1)];
      wv[j] = wg[min(tid + 256 * j, nx - 1)];
    }
#pragma unroll
    for (int i = 0; i < kRouterRows; i++)
#pragma unroll
      for (int u = 0; u < PR; u++)
        rw[i][u] = reinterpret_cast<const uint4*>(a.router + (int64_t)min(wave + 4 * i, rows - 1) * a.K)[min(lane + 64 * u, np - 1)];
    if (ahead) load(0, cur);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < XV; j++)
      if (tid + 256 * j < nx) ss = squares(xv[j], ss);
    ss = dh::wave_sum_uniform(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)a.hidden + a.eps);
#pragma unroll
    for (int j = 0; j < XV; j++) {
      const int i = tid + 256 * j;
      if (i < nx) planes[(i & 1) * np + (i >> 1)] = scaled(xv[j], inv, wv[j]);
    }
    __syncthreads();
    float sum[kRouterRows] = {};
#pragma unroll
    for (int u = 0; u < PR; u++) {
      const int p = lane + 64 * u;
      if (p >= np) continue;                             // (an infinite weight read again past the row's end, times nothing, would be no number)
      const float4 xa = planes[p], xb = planes[np + p];
#pragma unroll
      for (int i = 0; i < kRouterRows; i++) {
        const uint4 w = rw[i][u];
        float s = sum[i];
        s = fmaf(xa.x, dh::bf16_low(w.x), s); s = fmaf(xa.y, dh::bf16_high(w.x), s);
        s = fmaf(xa.z, dh::bf16_low(w.y), s); s = fmaf(xa.w, dh::bf16_high(w.y), s);
        s = fmaf(xb.x, dh::bf16_low(w.z), s); s = fmaf(xb.y, dh::bf16_high(w.z), s);
        s = fmaf(xb.z, dh::bf16_low(w.w), s); s = fmaf(xb.w, dh::bf16_high(w.w), s);
        sum[i] = s;
      }
    }
#pragma unroll
    for (int i = 0; i < kRouterRows; i++) {
      const float s = dh::wave_sum_uniform(sum[i]);
      if (lane == 0) {
        logits_s[wave + 4 * i] = s;
        if (blockIdx.x == 0 && wave + 4 * i < rows) a.z[wave + 4 * i] = s;
      }
    }
    __syncthreads();
    z = logits_s;
    if (wave == 0) choose(z, a.E, a.top, ids, zs);
    __syncthreads();
    if (!ahead) load(0, cur);
  } else {
    float ss = 0.f;
    for (int i = tid; i < (a.K >> 2); i += 256) ss = squares(xg[i], ss);
    ss = dh::wave_sum_uniform(ss);
    if (lane == 0) red[wave] = ss;
    if (wave == 0) choose(z, a.E, a.top, ids, zs);
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)a.hidden + a.eps);
    for (int i = tid; i < (a.K >> 2); i += 256) planes[(i & 1) * np + (i >> 1)] = scaled(xg[i], inv, wg[i]);
    __syncthreads();
    load(0, cur);
  }
  float acc[2] = {0.f, 0.f};
  int st = 0, it = 0;
  for (int unit = 0; unit < iters * nstages; unit++) {
    if (unit + 1 < iters * nstages) load(unit + 1, nxt);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int p = min(lane + 64 * (u + U * st), np - 1);
      const float4 xa = planes[p], xb = planes[np + p];
#pragma unroll
      for (int r = 0; r < 2; r++) {
        const uint4 w = cur[r][u];
        float s = acc[r];
        s = fmaf(xa.x, dh::bf16_low(w.x), s); s = fmaf(xa.y, dh::bf16_high(w.x), s);
        s = fmaf(xa.z, dh::bf16_low(w.y), s); s = fmaf(xa.w, dh::bf16_high(w.y), s);
        s = fmaf(xb.x, dh::bf16_low(w.z), s); s = fmaf(xb.y, dh::bf16_high(w.z), s);
        s = fmaf(xb.z, dh::bf16_low(w.w), s); s = fmaf(xb.w, dh::bf16_high(w.w), s);
        acc[r] = s;
      }
    }
    if (++st == nstages) {
      const float g = dh::wave_sum_uniform(acc[0]), u = dh::wave_sum_uniform(acc[1]);
      const int col = (it * (int)gridDim.x + (int)blockIdx.x) * 4 + wave;
      if (lane == 0 && col < total) {
        if (col >= a.top * a.ff) {
          a.act[col] = dh::clamped_glu(g, u, a.shared_limit) * sigmoid_f(z[a.E]);
        } else {
          const float s = sigmoid_f(zs[col / a.ff]);
          a.act[col] = dh::clamped_glu(s * g, s * u, a.limit);
        }
      }
      acc[0] = acc[1] = 0.f;
      st = 0;
      it++;
    }
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int u = 0; u < U; u++) cur[r][u] = nxt[r][u];
  }
}

// out[n] += ls[n] * [chosen down rows | shared down row] . act; a wave takes R rows at a time.  A chain of trips to memory (hidden 1024, four
// of 16 experts: 4 MB): every wave chooses for itself and requests its first weights at once, the row goes to LDS meanwhile, and an output's old
// value and scale come with its weights (5.7 -> 4.9 us; the same for the up kernel gave nothing, 7.0).
template <int R, int U>
__global__ __launch_bounds__(256) void experts_down_kernel(const StepArgs a, int iters) {
  extern __shared__ __align__(16) float4 planes[];       // [2][total / 8]
  __shared__ int ids[4][kMaxTop];
  __shared__ float zs[4][kMaxTop];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int np = (a.top * a.ff + a.shared_ff) >> 3, npe = a.ff >> 3, routed = a.top * npe;
  const int nstages = (np + 64 * U - 1) / (64 * U);
  // at / npe is at * ceil(2^32 / npe) >> 32, exact while at * npe stays below 2^32 (both are at most 4096; npe is 8 at least)
  const uint32_t npe_inverse = (uint32_t)(0xffffffffu / (uint32_t)npe + 1u);
  // the first pieces of the row are requested in front of the choice and the first weights (past the end the last piece again)
  const float4* act = reinterpret_cast<const float4*>(a.act);
  const int last = 2 * np - 1, i0 = min(tid, last), i1 = min(tid + 256, last), i2 = min(tid + 512, last), i3 = min(tid + 768, last);
  const float4 v0 = act[i0], v1 = act[i1], v2 = act[i2], v3 = act[i3];
  choose(a.z, a.E, a.top, ids[wave], zs[wave]);
  __builtin_amdgcn_wave_barrier();
  uint4 cur[R][U], nxt[R][U];
  auto first_row = [&](int it) { return ((it * (int)gridDim.x + (int)blockIdx.x) * 4 + wave) * R; };
  auto load = [&](int unit, uint4 (&dst)[R][U]) {
    const int it = unit / nstages, st = unit - it * nstages, row0 = first_row(it);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int p = lane + 64 * (u + U * st), at = min(p, np - 1);
      const int e = min((int)__umulhi((uint32_t)at, npe_inverse), a.top - 1);
      const bool chosen = at < routed;
      const uint16_t* w = chosen ? a.down + (int64_t)ids[wave][e] * a.hidden * a.ff + 8 * (at - e * npe) : a.shared_down + 8 * (at - routed);
      const int64_t ld = chosen ? a.ff : a.shared_ff;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint4 x = dh::stream_load_16(reinterpret_cast<const uint4*>(w + (int64_t)min(row0 + r, a.hidden - 1) * ld));
        dst[r][u] = p < np ? x : make_uint4(0, 0, 0, 0);
      }
    }
  };
  // the output row's old values and scales come with its first weights
  struct Terms {
    float scale[R], out[R];
  };
  Terms cur_terms, nxt_terms;
  auto load_terms = [&](int unit, Terms& t) {
    if (unit % nstages) return;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int n = min(first_row(unit / nstages) + r, a.hidden - 1);
      t.scale[r] = a.ls ? a.ls[n] : 1.f;
      t.out[r] = a.out[n];
    }
  };
  load(0, cur);
  load_terms(0, cur_terms);
  auto put = [&](int i, const float4& x) { planes[(i & 1) * np + (i >> 1)] = x; };
  put(i0, v0); put(i1, v1); put(i2, v2); put(i3, v3);
  for (int i = tid + 1024; i <= last; i += 256) put(i, act[i]);
  __syncthreads();
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = 0.f;
  int st = 0, it = 0;
  for (int unit = 0; unit < iters * nstages; unit++) {
    nxt_terms = cur_terms;
    if (unit + 1 < iters * nstages) {
      load(unit + 1, nxt);
      load_terms(unit + 1, nxt_terms);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int p = min(lane + 64 * (u + U * st), np - 1);
      const float4 xa = planes[p], xb = planes[np + p];
#pragma unroll
      for (int r = 0; r < R; r++) {
        const uint4 w = cur[r][u];
        float s = acc[r];
        s = fmaf(xa.x, dh::bf16_low(w.x), s); s = fmaf(xa.y, dh::bf16_high(w.x), s);
        s = fmaf(xa.z, dh::bf16_low(w.y), s); s = fmaf(xa.w, dh::bf16_high(w.y), s);
        s = fmaf(xb.x, dh::bf16_low(w.z), s); s = fmaf(xb.y, dh::bf16_high(w.z), s);
        s = fmaf(xb.z, dh::bf16_low(w.w), s); s = fmaf(xb.w, dh::bf16_high(w.w), s);
        acc[r] = s;
      }
    }
    if (++st == nstages) {
      const int row0 = first_row(it);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float v = dh::wave_sum_uniform(acc[r]);
        acc[r] = 0.f;
        const int n = row0 + r;
        if (lane == 0 && n < a.hidden) a.out[n] = fmaf(cur_terms.scale[r], v, cur_terms.out[r]);
      }
      st = 0;
      it++;
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int u = 0; u < U; u++) cur[r][u] = nxt[r][u];
    cur_terms = nxt_terms;
  }
}

// ------------------------------------------------------------------ portions

// A token's choices from its logits, by one wave.
__device__ __forceinline__ void route_token(const float* z, int t, int E, int top, int shared, int* id_s, float* z_s, int* __restrict__ ids,
                                            float* __restrict__ weights, float* __restrict__ sg) {
  const int lane = threadIdx.x & 63;
  choose(z, E, top, id_s, z_s);
  __builtin_amdgcn_wave_barrier();
  if (lane < top) {
    ids[(int64_t)t * top + lane] = id_s[lane];
    weights[(int64_t)t * top + lane] = sigmoid_f(z_s[lane]);
  }
  if (shared && lane == 0) sg[t] = sigmoid_f(z[E]);
}

// Logits of sixteen tokens, up to 16 NT of them each, and the tokens' choices.  Few columns over a long k are one trip to memory and a short product: each of
// the waves takes every sixteenth 32 of k straight from memory into its fragments of v_mfma_f32_16x16x32_bf16, four of them requested together, and
// the waves' sums meet in LDS in wave order.  What the places need goes out with the choices: slot, a choice's rank among the group's of its expert (in any
// order), and counts [groups][E].  us, 1531 rows of 2048, 16 experts and a shared one: 8.1, against 6.1 + 5.3 + 4.8 for a product
// with k in slices, the slices' sum and the choices; 40 rows of 1024 8 against 6.6 + 3.3.
constexpr int kRouterLogits = 32, kRouterWaves = 16;
template <int NT>
__global__ __launch_bounds__(64 * kRouterWaves) void experts_router_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ router, int K, int T, int E, int top,
                                                             int shared, int* __restrict__ ids, float* __restrict__ weights, float* __restrict__ sg,
                                                             int* __restrict__ slot, int* __restrict__ counts) {
  constexpr int WAVES = kRouterWaves, AHEAD = 64 / WAVES, ROW = 16 * NT + 4;
  __shared__ __align__(16) float sums[WAVES][16][ROW];
  __shared__ int id_s[WAVES][kMaxTop];
  __shared__ float z_s[WAVES][kMaxTop];
  __shared__ int count[kRouterLogits];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, t0 = 16 * blockIdx.x, n = E + shared;
  // a lane's row of either operand and its eight of every 32 k
  const uint16_t* a = h + (int64_t)min(t0 + (lane & 15), T - 1) * K + 8 * (lane >> 4);
  const uint16_t* b[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) b[j] = router + (int64_t)min(16 * j + (lane & 15), n - 1) * K + 8 * (lane >> 4);
  dh::f32x4_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) acc[j] = dh::f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 32 * wave; k0 < K; k0 += 32 * WAVES * AHEAD) {
    dh::bf16x8_t fa[AHEAD], fb[AHEAD][NT];
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      const int at = min(k0 + 32 * WAVES * u, K - 32);
      fa[u] = *reinterpret_cast<const dh::bf16x8_t*>(a + at);
#pragma unroll
      for (int j = 0; j < NT; j++) fb[u][j] = *reinterpret_cast<const dh::bf16x8_t*>(b[j] + at);
    }
    __builtin_amdgcn_sched_barrier(0);                 // (left alone the compiler requests each when it is due)
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      if (k0 + 32 * WAVES * u >= K) {                  // (both: an infinite weight times nothing is no number)
        fa[u] = dh::bf16x8_t{};
#pragma unroll
        for (int j = 0; j < NT; j++) fb[u][j] = dh::bf16x8_t{};
      }
#pragma unroll
      for (int j = 0; j < NT; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[u], fb[u][j], acc[j], 0, 0, 0);
    }
  }
  // accumulator element e of a lane: token 4 (lane / 16) + e, logit lane % 16
#pragma unroll
  for (int j = 0; j < NT; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) sums[wave][4 * (lane >> 4) + e][16 * j + (lane & 15)] = acc[j][e];
  __syncthreads();
  for (int i = tid; i < 16 * 16 * NT; i += 64 * WAVES) {
    const int t = i / (16 * NT), c = i % (16 * NT);
    float z = sums[0][t][c];
#pragma unroll
    for (int w = 1; w < WAVES; w++) z += sums[w][t][c];
    sums[0][t][c] = z;                                 // (read by this thread alone)
  }
  if (tid < kRouterLogits) count[tid] = 0;
  __syncthreads();
  if (t0 + wave < T) {
    route_token(sums[0][wave], t0 + wave, E, top, shared, id_s[wave], z_s[wave], ids, weights, sg);
    if (lane < top) slot[(int64_t)(t0 + wave) * top + lane] = atomicAdd(&count[id_s[wave][lane]], 1);
  }
  __syncthreads();
  if (tid < E) counts[(int64_t)blockIdx.x * E + tid] = count[tid];
}

// One wave per token.
__global__ __launch_bounds__(256) void experts_route_kernel(const float* __restrict__ z, int64_t ld_z, int T, int E, int top, int shared,
                                                            int* __restrict__ ids, float* __restrict__ weights, float* __restrict__ sg) {
  __shared__ int id_s[4][kMaxTop];
  __shared__ float z_s[4][kMaxTop];
  const int wave = threadIdx.x >> 6, t = blockIdx.x * 4 + wave;
  if (t < T) route_token(z + (int64_t)t * ld_z, t, E, top, shared, id_s[wave], z_s[wave], ids, weights, sg);
}

// Sorted places of the router kernel's choices, by workgroups of 64 tokens (four of its groups): every one of them adds up the groups' counts of every
// expert, in all and in front of its own tokens.  A few short steps on many compute units (6124 choices of 16 experts 5.1 us, 160 choices 3.5), where
// experts_sort_kernel takes one unit through all choices twice (9.9 and 5.5); it stays for more groups than a workgroup adds up in passing, more
// experts, and choices that do not come in groups.
constexpr int kPlacedGroups = 256;                     // 4096 tokens
__global__ __launch_bounds__(256) void experts_place_kernel(const int* __restrict__ ids, const float* __restrict__ weights, const int* __restrict__ counts, int n, int top,
                                                            int E, int groups, int tile_rows, int max_tiles, int* __restrict__ off, int* __restrict__ slot,
                                                            int* __restrict__ row_token, float* __restrict__ row_weight, int* __restrict__ tiles) {
  constexpr int GROUPS = 4, CHOICES = 16 * GROUPS, BATCH = 4;        // of a workgroup; CHOICES for each of a token's `top`
  __shared__ int part[2][256];                         // sums of a thread's groups: all of them, and those in front
  __shared__ int at[GROUPS][kRouterLogits];            // where a group's rows of an expert begin
  const int tid = threadIdx.x, g0 = GROUPS * blockIdx.x, i0 = CHOICES * top * blockIdx.x, mine = min(CHOICES * top, n - i0);
  const int shift = E <= 16 ? 4 : 5, parts = 256 >> shift, e = tid & ((1 << shift) - 1);
  int id[BATCH], rank[BATCH];
  float w[BATCH];
  auto read = [&](int j) {
#pragma unroll
    for (int k = 0; k < BATCH; k++) {
      const int i = i0 + min(j + 256 * k, mine - 1);
      id[k] = ids[i];
      rank[k] = slot[i];
      w[k] = weights[i];
    }
  };
  read(tid);
  int all = 0, front = 0;
#pragma unroll 4
  for (int g = tid >> shift; g < groups; g += parts) {
    const int c = e < E ? counts[g * E + e] : 0;
    all += c;
    front += g < g0 ? c : 0;
  }
  part[0][tid] = all;
  part[1][tid] = front;
  __syncthreads();
  if (tid < 64) {                                      // lane: an expert
    all = front = 0;
    if (tid < E)
      for (int k = 0; k < parts; k++) {
        all += part[0][tid + (k << shift)];
        front += part[1][tid + (k << shift)];
      }
    const int my_tiles = (all + tile_rows - 1) / tile_rows;
    int rows = all, upto = my_tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(rows, o, 64), b = __shfl_up(upto, o, 64);
      if (tid >= o) {
        rows += a;
        upto += b;
      }
    }
    const int first = rows - all;
    int next = first + front;
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
      if (tid >= E) break;
      at[g][tid] = next;
      if (g0 + g < groups) next += counts[(g0 + g) * E + tid];
    }
    if (blockIdx.x == 0) {
      if (tid < E) off[tid] = first;
      if (tid == E - 1) off[E] = n;
      for (int k = 0; k < my_tiles; k++) {
        tiles[2 * (upto - my_tiles + k)] = tid;
        tiles[2 * (upto - my_tiles + k) + 1] = k * tile_rows;
      }
      for (int k = __shfl(upto, 63, 64) + tid; k < max_tiles; k += 64) tiles[2 * k] = -1;
    }
  }
  __syncthreads();
  for (int j = tid; j < mine; j += 256 * BATCH) {
    if (j != tid) read(j);
#pragma unroll
    for (int k = 0; k < BATCH; k++) {
      const int own = j + 256 * k, i = i0 + own;
      if (own >= mine) break;
      const int to = at[own / (16 * top)][id[k]] + rank[k];
      slot[i] = to;
      row_token[to] = i / top;
      row_weight[to] = w[k];
    }
  }
}

// Where the two kernels above stand in for a product, its slices' sum, the choices and the sort.  Every workgroup reads the whole router, and with more
// logits twice the accumulators' rows, where a product spreads a long k over the device; what the sort saves grows with the tokens.  Whole portions of 64
// wide experts in us, product and sort / these: 16 logits, 200 tokens, k 2048 36.7 / 33.6, 4096 56.5 / 55.8, 5120 64.2 / 66.5; 32 logits k 2048 42.8 / 41.7,
// 3072 51.1 / 55.1, 4096 58.9 / 63.0, with 4096 tokens 222.5 / 220.0 (17: 212.0 / 201.8); 64 logits, 200 tokens, k 256 22.7 / 31.7, 2048 43.5 / 48.9.
bool routes_itself(int logits, int K, int T) {
  return logits <= kRouterLogits && T <= 16 * kPlacedGroups && (K <= 2048 || (K <= 4096 && (logits <= 16 || T > 1024)));
}

// One workgroup: rows sorted by expert.  slot[i]: sorted place of choice i = token * top + k; row_token, row_weight by place.
__global__ __launch_bounds__(1024) void experts_sort_kernel(const int* __restrict__ ids, const float* __restrict__ weights, int n, int top,
                                                            int E, int tile_rows, int max_tiles, int* __restrict__ off, int* __restrict__ slot,
                                                            int* __restrict__ row_token, float* __restrict__ row_weight, int* __restrict__ tiles) {
  __shared__ int count[kMaxExperts];
  __shared__ int scan[kMaxExperts];
  __shared__ int tscan[kMaxExperts];
  const int tid = threadIdx.x;
  count[tid] = 0;
  __syncthreads();
  constexpr int BATCH = 8;                               // reads in flight per thread
  for (int i0 = tid; i0 < n; i0 += 1024 * BATCH) {
    int id[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; k++) id[k] = i0 + 1024 * k < n ? ids[i0 + 1024 * k] : -1;
#pragma unroll
    for (int k = 0; k < BATCH; k++)
      if (id[k] >= 0) atomicAdd(&count[id[k]], 1);
  }
  __syncthreads();
  const int mine = count[tid], my_tiles = (mine + tile_rows - 1) / tile_rows;
  scan[tid] = mine;
  tscan[tid] = my_tiles;
  __syncthreads();
  for (int o = 1; o < kMaxExperts; o <<= 1) {
    const int a = tid >= o ? scan[tid - o] : 0, b = tid >= o ? tscan[tid - o] : 0;
    __syncthreads();
    scan[tid] += a;
    tscan[tid] += b;
    __syncthreads();
  }
  const int first = scan[tid] - mine, first_tile = tscan[tid] - my_tiles, used = tscan[kMaxExperts - 1];
  if (tid < E) off[tid] = first;
  if (tid == E - 1) off[E] = n;
  for (int k = 0; k < my_tiles; k++) {
    tiles[2 * (first_tile + k)] = tid;
    tiles[2 * (first_tile + k) + 1] = k * tile_rows;
  }
  for (int k = used + tid; k < max_tiles; k += 1024) tiles[2 * k] = -1;
  count[tid] = first;                                    // next free place of the expert
  __syncthreads();
  for (int i0 = tid; i0 < n; i0 += 1024 * BATCH) {
    int id[BATCH];
    float w[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; k++) {
      const int i = i0 + 1024 * k;
      id[k] = i < n ? ids[i] : -1;
      w[k] = i < n ? weights[i] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < BATCH; k++) {
      const int i = i0 + 1024 * k;
      if (id[k] < 0) continue;
      const int at = atomicAdd(&count[id[k]], 1);        // any order inside a group: a row's results do not depend on its place
      slot[i] = at;
      row_token[at] = i / top;
      row_weight[at] = w[k];
    }
  }
}

// x[t] += ls * sum of the token's rows, then ls * the shared expert's row where that is not null (rounded as an epilogue with scale and residual
// does: a token has the same bits whether the products share a launch or not).  Four columns per thread.
__global__ __launch_bounds__(256) void experts_combine_kernel(const float* __restrict__ y, int64_t ld_y, const int* __restrict__ slot, int top,
                                                              const float* __restrict__ shared, const float* __restrict__ ls, float* __restrict__ x,
                                                              int64_t ld_x, int hidden) {
  const int t = blockIdx.x, i = 4 * (blockIdx.y * 256 + threadIdx.x);
  if (i >= hidden) return;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f), own = s;
  if (shared) own = *reinterpret_cast<const float4*>(shared + (int64_t)t * ld_y + i);
  for (int k = 0; k < top; k++) {
    const float4 v = *reinterpret_cast<const float4*>(y + (int64_t)slot[(int64_t)t * top + k] * ld_y + i);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  const float sv[4] = {s.x, s.y, s.z, s.w}, ov[4] = {own.x, own.y, own.z, own.w};
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if (i + e >= hidden) break;
    float* o = x + (int64_t)t * ld_x + i + e;
    const float f = ls ? ls[i + e] : 1.f;
    float v = fmaf(f, sv[e], *o);
    if (shared) v = fmaf(ov[e], f, 0.f) + v;
    *o = v;
  }
}

// The same where nothing is added behind it, and the rows normed for the product that reads them: one workgroup a row (at most 4096 columns, a multiple of
// four, x and ls aligned).  Against a launch of the norm's own, us: 1531 rows of 2048 18.9 + 5.6 -> 17.1, 40 of 1024 4.3 + 3.1 -> 4.8.  What a thread adds up one
// after the other is its pieces times the choices: whole portions of 16 tokens, apart / in one, 32 choices of 3072 columns 59.6 / 57.3, of 4096 66.9 / 68.1, of 8192 97.4
// / 112.3, 16 of 4096 60.4 / 60.2, of 6144 76.3 / 79.2, two of 8192 72.1 / 74.8.
template <bool BF16>
__global__ __launch_bounds__(256) void experts_combine_norm_kernel(const float* __restrict__ y, int64_t ld_y, const int* __restrict__ slot, int top,
                                                                   const float* __restrict__ shared, const float* __restrict__ ls, float* __restrict__ x,
                                                                   int64_t ld_x, int hidden, const float* __restrict__ norm, float eps, void* __restrict__ normed,
                                                                   int ld_normed) {
  __shared__ float red[4];
  const int t = blockIdx.x;
  const int* places = slot + (int64_t)t * top;
  float* row = x + (int64_t)t * ld_x;
  float4 out[dh::kMadePieces];
#pragma unroll
  for (int j = 0; j < dh::kMadePieces; j++) {
    const int i = 4 * (threadIdx.x + 256 * j);
    out[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= hidden) continue;
    const float4 old = *reinterpret_cast<const float4*>(row + i);
    float4 s = out[j], own = s, f = make_float4(1.f, 1.f, 1.f, 1.f);
    if (shared) own = *reinterpret_cast<const float4*>(shared + (int64_t)t * ld_y + i);
    if (ls) f = *reinterpret_cast<const float4*>(ls + i);
#pragma unroll 4
    for (int k = 0; k < top; k++) {
      const float4 v = *reinterpret_cast<const float4*>(y + (int64_t)places[k] * ld_y + i);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    auto sum = [&](float f, float s, float own, float old) {
      const float v = fmaf(f, s, old);
      return shared ? fmaf(own, f, 0.f) + v : v;
    };
    out[j] = make_float4(sum(f.x, s.x, own.x, old.x), sum(f.y, s.y, own.y, old.y), sum(f.z, s.z, own.z, old.z), sum(f.w, s.w, own.w, old.w));
    *reinterpret_cast<float4*>(row + i) = out[j];
  }
  dh::store_normed_row<BF16>(out, hidden, norm, eps, red, normed, (int64_t)t * ld_normed, ld_normed);
}
bool sums_in_passing(int hidden, int top) { return hidden <= 1024 * dh::kMadePieces && (int64_t)hidden * top <= 3 << 15; }

// Where a step's first kernel makes the logits too (20 are what its waves hold).  Four pieces of a row leave three workgroups to a compute unit's registers, and
// a fourth would wait for one of them to end; and what a launch saves is more than twenty rows' reading only where there are few workgroups or the rows are long.
// us, logits in a launch / in the kernel, four of the experts: 20 logits, 768 workgroups, k 256 12.3 / 12.1, 1536 15.8 / 15.1, 2048 17.0 / 15.8; 1024 workgroups,
// k 256 12.8 / 13.2, 512 13.2 / 13.3, 1024 14.3 / 13.5, 1536 16.8 / 20.0, 2048 18.2 / 20.7; 17 logits, 784 workgroups, k 1024 13.9 / 12.2, 2048 17.4 / 18.3;
// 16 logits, 1024 workgroups, k 256 12.8 / 12.7; 9 logits, 528 workgroups, k 1024 13.2 / 10.5, 2048 16.3 / 13.3.
bool router_beside(int logits, int K, int workgroups) {
  return logits <= 4 * kRouterRows && K <= 2048 && (workgroups <= 3 * dh::num_cus() || (K <= 1024 && (logits <= 16 || K >= 512)));
}

size_t up256(size_t n) { return (n + 255) / 256 * 256; }
bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check(const char* op, const dh_experts* s) {
  if (!s) return dh::fail(1, "[%s] null spec", op);
  if (s->hidden <= 0 || s->K < s->hidden || s->K % 64) return dh::fail(1, "[%s] hidden=%d in rows of %d (a multiple of 64)", op, s->hidden, s->K);
  if (s->experts <= 0 || s->experts > kMaxExperts || s->top <= 0 || s->top > kMaxTop || s->top > s->experts)
    return dh::fail(1, "[%s] %d of %d experts (at most %d of %d)", op, s->top, s->experts, kMaxTop, kMaxExperts);
  if (s->ff <= 0 || s->ff % 64 || s->shared_ff < 0 || s->shared_ff % 64) return dh::fail(1, "[%s] expert widths must be multiples of 64 (%d, shared %d)", op, s->ff, s->shared_ff);
  if (!s->d_router || !s->d_up || !s->d_down || !s->d_norm || (s->shared_ff && (!s->d_shared_up || !s->d_shared_down))) return dh::fail(1, "[%s] null pointer in the spec", op);
  if (!aligned(s->d_router) || !aligned(s->d_up) || !aligned(s->d_down) || !aligned(s->d_norm) || !aligned(s->d_shared_up) || !aligned(s->d_shared_down))
    return dh::fail(1, "[%s] weights must be 16-byte aligned", op);
  return 0;
}
int logits(const dh_experts* s) { return s->experts + (s->shared_ff ? 1 : 0); }

// Where a portion's intermediate rows lie in the workspace.
struct PortionSpace {
  size_t z, ids, weights, sg, off, slot, row_token, row_weight, tiles, act, shared_act, y, shared_y, end;
  int ld_z, ld_y, max_tiles, tile_rows;
};
PortionSpace portion_space(const dh_experts* s, int operand, int T) {
  PortionSpace p{};
  const size_t n = (size_t)T * s->top, elem = operand == DH_F32 ? 4 : 2;
  p.ld_z = (logits(s) + 3) / 4 * 4;
  p.ld_y = (s->hidden + 3) / 4 * 4;
  p.tile_rows = dh::expert_tile_rows(operand, (int)n, s->experts);
  p.max_tiles = (int)(n / p.tile_rows + std::min<size_t>(n, s->experts));
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t r = at; at += up256(bytes); return r; };
  p.z = take((size_t)T * p.ld_z * 4);
  p.ids = take(n * 4); p.weights = take(n * 4); p.sg = take((size_t)T * 4);
  p.off = take((size_t)(s->experts + 1) * 4); p.slot = take(n * 4); p.row_token = take(n * 4); p.row_weight = take(n * 4);
  p.tiles = take((size_t)p.max_tiles * 8);
  p.act = take(n * s->ff * elem);
  p.shared_act = take((size_t)T * s->shared_ff * elem);
  p.y = take(n * p.ld_y * 4);
  p.shared_y = take(s->shared_ff && operand == DH_BF16 ? (size_t)T * p.ld_y * 4 : 0);
  p.end = at;
  return p;
}

// Sizes of a portion's four products: routed and shared, gate and up (glu) or down.
dh::ExpertProduct routed_product(const dh_experts* s, const PortionSpace& p, int T, bool glu) {
  dh::ExpertProduct r{};
  r.M = T * s->top; r.N = glu ? 2 * s->ff : s->hidden; r.lda = r.ldw = r.K = glu ? s->K : s->ff; r.ld_out = glu ? s->ff : p.ld_y;
  r.rows.source_rows = T; r.rows.w_stride = (int64_t)r.N * r.K; r.rows.max_tiles = p.max_tiles; r.rows.tile_rows = p.tile_rows; r.rows.limit = s->limit;
  return r;
}
dh::ExpertProduct shared_product(const dh_experts* s, const PortionSpace& p, int T, bool glu) {
  dh::ExpertProduct r{};
  r.M = T; r.N = glu ? 2 * s->shared_ff : s->hidden; r.lda = r.ldw = r.K = glu ? s->K : s->shared_ff; r.ld_out = glu ? s->shared_ff : p.ld_y;
  r.rows.limit = s->shared_limit;
  return r;
}
bool together(const dh_experts* s, int operand, const PortionSpace& p, int T, bool glu) {
  return s->shared_ff > 0 && operand == DH_BF16 && dh::experts_together(routed_product(s, p, T, glu), shared_product(s, p, T, glu), glu);
}

// The norm of the rows a portion leaves, for the product that reads them next, or nothing; done: the last launch made it.
struct NextNorm {
  const float* weight = nullptr;
  float eps = 0.f;
  void* normed = nullptr;
  int ld = 0;
  bool* done = nullptr;
};
int prefill(const char* op, const dh_experts* spec, const void* d_h, int operand, float* d_x, int ld_x, void* d_workspace, int T, const NextNorm& next);

}  // namespace

extern "C" {

size_t dh_experts_step_workspace_bytes(const dh_experts* s) {
  if (!s) return 256;
  return up256((size_t)logits(s) * 4) + up256(((size_t)s->top * s->ff + s->shared_ff) * 4);
}

int dh_experts_step(const dh_experts* spec, float* d_x, void* d_workspace) {
  const char* op = "dh_experts_step";
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, spec)) return rc;
  if (!d_x || !d_workspace) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_x) || !aligned(d_workspace)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  const int64_t total = (int64_t)spec->top * spec->ff + spec->shared_ff;
  if (spec->K > 32768 || total > 32768) return dh::fail(1, "[%s] rows of %d and %lld elements: at most 32768 fit one workgroup", op, spec->K, (long long)total);
  float* z = static_cast<float*>(d_workspace);
  float* act = reinterpret_cast<float*>(static_cast<char*>(d_workspace) + up256((size_t)logits(spec) * 4));
  StepArgs a{};
  a.x = d_x; a.norm = spec->d_norm; a.z = z; a.router = static_cast<const uint16_t*>(spec->d_router);
  a.up = static_cast<const uint16_t*>(spec->d_up); a.down = static_cast<const uint16_t*>(spec->d_down);
  a.shared_up = static_cast<const uint16_t*>(spec->d_shared_up); a.shared_down = static_cast<const uint16_t*>(spec->d_shared_down);
  a.ls = spec->d_layer_scale; a.act = act; a.out = d_x;
  a.hidden = spec->hidden; a.K = spec->K; a.E = spec->experts; a.top = spec->top; a.ff = spec->ff; a.shared_ff = spec->shared_ff;
  a.eps = spec->eps; a.limit = spec->limit; a.shared_limit = spec->shared_limit;
  static bool attr_set = false;
  if (!attr_set) {
    for (const void* k : {reinterpret_cast<const void*>(experts_up_kernel<4, 0>), reinterpret_cast<const void*>(experts_down_kernel<1, 8>)})
      DH_CHECK_HIP(op, hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 32768 * 4));
    attr_set = true;
  }
  auto plan = [&](int64_t units, int64_t k, int* iters) {
    const int64_t most = (k <= 8192 ? 4 : k <= 16384 ? 2 : 1) * (int64_t)dh::num_cus();
    *iters = (int)std::max<int64_t>(1, dh::ceil_div(units, most));
    return dim3((unsigned)dh::ceil_div(units, *iters));
  };
  int iters = 1;
  dim3 grid = plan(dh::ceil_div(total, 4), spec->K, &iters);
  const bool with_router = router_beside(logits(spec), spec->K, (int)grid.x);
  if (!with_router)
    if (int rc = dh_dense_gemv(d_x, spec->d_norm, spec->hidden, spec->eps, spec->d_router, spec->K, logits(spec), spec->K, 1.f, nullptr, nullptr, z,
                               logits(spec), nullptr, DH_ACT_NONE))
      return rc;
  auto up = !with_router ? experts_up_kernel<4, 0> : spec->K <= 1024 ? experts_up_kernel<4, 2> : experts_up_kernel<4, 4>;
  hipLaunchKernelGGL(up, grid, dim3(256), (size_t)spec->K * 4, dh::stream(), a, iters);
  DH_CHECK_LAUNCH(op);
  grid = plan(dh::ceil_div(spec->hidden, 4), total, &iters);
  hipLaunchKernelGGL((experts_down_kernel<1, 8>), grid, dim3(256), (size_t)total * 4, dh::stream(), a, iters);
  DH_CHECK_LAUNCH(op);
  return 0;
}

size_t dh_experts_prefill_workspace_bytes(const dh_experts* s, int operand, int T) { return s && T > 0 ? portion_space(s, operand, T).end : 256; }

int dh_experts_prefill_layout(const dh_experts* spec, int operand, int T, int num_cus, int64_t* out3) {
  const char* op = "dh_experts_prefill_layout";
  if (int rc = check(op, spec)) return rc;
  if (!out3 || T <= 0 || (int64_t)T * spec->top > (1 << 24) || (operand != DH_BF16 && operand != DH_F32))
    return dh::fail(1, "[%s] T=%d, dtype %d, or no place for the result", op, T, operand);
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  const PortionSpace p = portion_space(spec, operand, T);
  out3[0] = p.tile_rows;
  out3[1] = together(spec, operand, p, T, true);
  out3[2] = together(spec, operand, p, T, false);
  dh::plan_end();
  return 0;
}

int dh_experts_prefill(const dh_experts* spec, const void* d_h, int operand, float* d_x, int ld_x, void* d_workspace, int T) {
  return prefill("dh_experts_prefill", spec, d_h, operand, d_x, ld_x, d_workspace, T, NextNorm{});
}

int dh_experts_prefill_normed(const dh_experts* spec, const void* d_h, int operand, float* d_x, int ld_x, void* d_workspace, int T, const float* d_norm_weight,
                              float eps, void* d_normed, int ld_normed) {
  const char* op = "dh_experts_prefill_normed";
  DH_REQUIRE_INIT(op);
  if (!d_norm_weight || !d_normed) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_norm_weight) || !aligned(d_normed)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  if (spec && (ld_normed < spec->hidden || !(eps >= 0.f))) return dh::fail(1, "[%s] normed rows of %d do not hold %d elements, or eps is negative", op, ld_normed, spec->hidden);
  bool done = false;
  if (int rc = prefill(op, spec, d_h, operand, d_x, ld_x, d_workspace, T, NextNorm{d_norm_weight, eps, d_normed, ld_normed, &done})) return rc;
  return done ? 0 : dh_rmsnorm_rows(d_x, ld_x, nullptr, d_norm_weight, d_normed, operand, ld_normed, T, spec->hidden, eps);
}

}  // extern "C"

namespace {
int prefill(const char* op, const dh_experts* spec, const void* d_h, int operand, float* d_x, int ld_x, void* d_workspace, int T, const NextNorm& next) {
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, spec)) return rc;
  if (T <= 0 || ld_x < spec->hidden) return dh::fail(1, "[%s] %d rows %d apart", op, T, ld_x);
  if (operand != DH_BF16 && operand != DH_F32) return dh::fail(1, "[%s] activations must be bf16 or f32, got dtype %d", op, operand);
  if (!d_h || !d_x || !d_workspace) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_h) || !aligned(d_workspace)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  if ((int64_t)T * spec->top > (1 << 24)) return dh::fail(1, "[%s] %d tokens are too many for one portion", op, T);
  if (operand == DH_BF16 && T > 1 && (int64_t)T * spec->K >= (int64_t)1 << 31) {
    // gathered rows are addressed by 32-bit byte offsets: more than 4 GB of them go in two portions
    const int half = T / 2;
    if (int rc = prefill(op, spec, d_h, operand, d_x, ld_x, d_workspace, half, NextNorm{})) return rc;
    return prefill(op, spec, static_cast<const uint16_t*>(d_h) + (int64_t)half * spec->K, operand, d_x + (int64_t)half * ld_x, ld_x, d_workspace, T - half, NextNorm{});
  }
  const PortionSpace p = portion_space(spec, operand, T);
  char* w = static_cast<char*>(d_workspace);
  auto f32 = [&](size_t at) { return reinterpret_cast<float*>(w + at); };
  auto i32 = [&](size_t at) { return reinterpret_cast<int*>(w + at); };
  const int n = T * spec->top;
  const int shared_logit = spec->shared_ff > 0 ? 1 : 0, groups = (int)dh::ceil_div(T, 16);
  if (operand == DH_BF16 && routes_itself(logits(spec), spec->K, T)) {
    auto kern = logits(spec) <= 16 ? experts_router_kernel<1> : experts_router_kernel<2>;
    int* counts = i32(p.z);                            // (no logits go to memory)
    hipLaunchKernelGGL(kern, dim3(groups), dim3(64 * kRouterWaves), 0, dh::stream(), static_cast<const uint16_t*>(d_h),
                       static_cast<const uint16_t*>(spec->d_router), spec->K, T, spec->experts, spec->top, shared_logit, i32(p.ids), f32(p.weights), f32(p.sg),
                       i32(p.slot), counts);
    DH_CHECK_LAUNCH(op);
    hipLaunchKernelGGL(experts_place_kernel, dim3((unsigned)dh::ceil_div(groups, 4)), dim3(256), 0, dh::stream(), i32(p.ids), f32(p.weights), counts, n, spec->top,
                       spec->experts, groups, p.tile_rows, p.max_tiles, i32(p.off), i32(p.slot), i32(p.row_token), f32(p.row_weight), i32(p.tiles));
    DH_CHECK_LAUNCH(op);
  } else {
    if (int rc = dh_dense_matmul(d_h, operand, spec->K, spec->d_router, spec->K, T, logits(spec), spec->K, 1.f, nullptr, nullptr, f32(p.z), p.ld_z,
                                 logits(spec), nullptr, 0, 0, DH_ACT_NONE))
      return rc;
    hipLaunchKernelGGL(experts_route_kernel, dim3((unsigned)dh::ceil_div(T, 4)), dim3(256), 0, dh::stream(), f32(p.z), (int64_t)p.ld_z, T, spec->experts,
                       spec->top, shared_logit, i32(p.ids), f32(p.weights), f32(p.sg));
    DH_CHECK_LAUNCH(op);
    hipLaunchKernelGGL(experts_sort_kernel, dim3(1), dim3(1024), 0, dh::stream(), i32(p.ids), f32(p.weights), n, spec->top, spec->experts, p.tile_rows,
                       p.max_tiles, i32(p.off), i32(p.slot), i32(p.row_token), f32(p.row_weight), i32(p.tiles));
    DH_CHECK_LAUNCH(op);
  }
  const uint16_t *up = static_cast<const uint16_t*>(spec->d_up), *down = static_cast<const uint16_t*>(spec->d_down);
  const uint16_t *shared_up = static_cast<const uint16_t*>(spec->d_shared_up), *shared_down = static_cast<const uint16_t*>(spec->d_shared_down);
  const bool shared = spec->shared_ff > 0, up_pair = together(spec, operand, p, T, true), down_pair = together(spec, operand, p, T, false);
  // gate and up products; the shared expert's beside the routed ones' or behind them
  dh::ExpertProduct routed = routed_product(spec, p, T, true), own = shared_product(spec, p, T, true);
  routed.A = own.A = d_h; routed.W = up; routed.out = w + p.act; own.W = shared_up; own.out = w + p.shared_act;
  routed.rows.tiles = i32(p.tiles); routed.rows.group_off = i32(p.off); routed.rows.row_index = i32(p.row_token); routed.rows.factor = f32(p.row_weight);
  routed.rows.factor_in = true; own.rows.factor = f32(p.sg);
  auto glu = [&](const dh::ExpertProduct& g) {
    return dh::experts_glu(op, g.rows, g.A, operand, g.lda, g.W, g.ldw, g.M, g.N, g.K, g.out, operand, g.ld_out);
  };
  if (int rc = up_pair ? dh::experts_pair(op, routed, own, true) : glu(routed)) return rc;
  auto shared_gate_up = [&] { return up_pair ? 0 : glu(own); };
  // down products: together, the shared expert's waits in the workspace until the routed ones' sum has reached x
  dh::ExpertProduct routed_down = routed_product(spec, p, T, false), own_down = shared_product(spec, p, T, false);
  routed_down.A = w + p.act; routed_down.W = down; routed_down.out = f32(p.y); routed_down.rows.tiles = i32(p.tiles); routed_down.rows.group_off = i32(p.off);
  own_down.A = w + p.shared_act; own_down.W = shared_down; own_down.out = f32(p.shared_y);
  if (down_pair) {
    if (int rc = shared_gate_up()) return rc;
    if (int rc = dh::experts_pair(op, routed_down, own_down, false)) return rc;
  } else {
    if (int rc = dh::experts_down(op, routed_down.rows, w + p.act, operand, spec->ff, down, spec->ff, spec->hidden, spec->ff, f32(p.y), p.ld_y)) return rc;
  }
  if (next.weight && (!shared || down_pair) && spec->hidden % 4 == 0 && sums_in_passing(spec->hidden, spec->top) && ld_x % 4 == 0 && aligned(d_x) &&
      aligned(spec->d_layer_scale)) {
    auto kern = operand == DH_BF16 ? experts_combine_norm_kernel<true> : experts_combine_norm_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(T), dim3(256), 0, dh::stream(), f32(p.y), (int64_t)p.ld_y, i32(p.slot), spec->top, down_pair ? f32(p.shared_y) : nullptr,
                       spec->d_layer_scale, d_x, (int64_t)ld_x, spec->hidden, next.weight, next.eps, next.normed, next.ld);
    DH_CHECK_LAUNCH(op);
    *next.done = true;
    return 0;
  }
  hipLaunchKernelGGL(experts_combine_kernel, dim3(T, (unsigned)dh::ceil_div(spec->hidden, 1024)), dim3(256), 0, dh::stream(), f32(p.y), (int64_t)p.ld_y,
                     i32(p.slot), spec->top, down_pair ? f32(p.shared_y) : nullptr, spec->d_layer_scale, d_x, (int64_t)ld_x, spec->hidden);
  DH_CHECK_LAUNCH(op);
  if (shared && !down_pair) {
    if (int rc = shared_gate_up()) return rc;
    return dh_dense_matmul_scaled(w + p.shared_act, operand, spec->shared_ff, shared_down, spec->shared_ff, T, spec->hidden, spec->shared_ff, 1.f,
                                  nullptr, spec->d_layer_scale, d_x, d_x, ld_x, spec->hidden, nullptr, 0, 0, DH_ACT_NONE);
  }
  return 0;
}

}  // namespace
