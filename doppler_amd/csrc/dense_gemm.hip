// Matrix products with dense bf16 weights for several activation rows (prefill).
//
//   bf16 activations   v_mfma_f32_32x32x16_bf16, f32 accumulation
//   f16 activations    the same with f16 weights, v_mfma_f32_32x32x16_f16 (products of rows an f16 cache holds)
//   f32 activations    each the sum of three bf16, which makes every product exact, v_mfma_f32_32x32x16_bf16 (gemm_split.h)
//
// Weights [N][ldw] and activations [M][lda] are both read along k; K is a multiple of 64, which the owner of the buffers
// reaches with zero padding.  16-bit operands: gemm_wide.h (tiles of 256 x 256 down to 64 x 64, straight from memory into LDS).
// 32-bit: tiles of 128 x 128 down to 32 x 64, the same way; products of experts, of one step, and of rows out of reach go
// through registers, 32 k at a time, to v_mfma_f32_32x32x2_f32 on the weights widened (exactly) to f32.
//
// The epilogue serves two outputs, because the projections that read one normalised row are stored as one
// stacked matrix: columns below n_first are (alpha * acc + bias) * column scale (+ residual) in f32, columns from n_first
// on are act(alpha * acc), written in the operand type of the product that reads them.
//
// Experts (dh_experts_*): the GROUPED forms take rows that are sorted by expert.  A table of row tiles names every tile's
// expert and first row; a tile gathers its activation rows by index, multiplies them by its own expert's weights and
// leaves when the table has ended.  The GLU forms read matrices whose gate and up rows alternate in blocks of 32, so
// that a wave's two neighbouring accumulator tiles hold the gate and the up value of the same column in the same lane;
// the epilogue clamps, gates and multiplies them and writes one column per pair.
//
// A grid of too few tiles for the device cuts k into slices instead (grid.y): every slice leaves its raw sums in the
// library's split-K workspace and a second launch adds them in slice order and runs the epilogue.
#include <algorithm>
#include <type_traits>

#include "dense_device.h"
#include "experts.h"
#include "gemm_split.h"

namespace {

using dh::bf16x8_t;
using dh::f16x8_t;
using dh::f32x16_t;
using dh::f32x4_t;
using dh::u32x4_t;

struct GemmArgs {
  const void* A;          // [M][lda], bf16 or f32
  const uint16_t* W;      // [N][ldw] bf16
  int64_t lda, ldw;
  int M, N, K;
  float alpha;
  const float* bias;      // [n_first] or null
  const float* residual;  // [M][ldc] or null (may be C)
  const float* col_scale; // [n_first] or null
  float* C;
  int ldc;
  int n_first;
  void* C2;               // [M][ldc2]
  int ldc2;
  int c2_dtype, act;
  int tiles_m, tiles_n;
  float* parts;           // [slices][M][N] raw sums instead of the outputs, or null
  int k_slice;            // k extent of a slice (a multiple of 64); K when there is one
  dh::ExpertRows rows;    // GROUPED and GLU forms
  // the first output's rows normed as well, where a reduce launch holds them whole (done: it did), or null
  const float* norm_weight;
  float norm_eps;
  void* normed;           // [M][ld_normed]
  int normed_dtype, ld_normed;
  bool* norm_done;
};

// Second outputs a kernel is compiled for: none (the first without or with a residual), one activation, or whatever the arguments say.
constexpr int kNoSecond = -2, kAnyAct = -3, kResidual = -4;
constexpr bool only_first(int act) { return act == kNoSecond || act == kResidual; }

__device__ __forceinline__ void put_c2(const GemmArgs& a, int64_t at, float v) {
  if (a.c2_dtype == DH_BF16) static_cast<uint16_t*>(a.C2)[at] = dh::f32_to_bf16_bits(v);
  else if (a.c2_dtype == DH_F16) static_cast<_Float16*>(a.C2)[at] = (_Float16)v;
  else static_cast<float*>(a.C2)[at] = v;
}

// The two outputs of one element; what the first adds and multiplies in is requested before anything is stored (see below).
struct PutTerms {
  float bias, scale, residual;
};
__device__ __forceinline__ bool has_terms(const GemmArgs& a) { return a.bias || a.col_scale || a.residual; }
__device__ __forceinline__ PutTerms put_terms(const GemmArgs& a, int m, int n) {
  PutTerms t{0.f, 1.f, 0.f};
  if (n < a.n_first) {
    if (a.bias) t.bias = a.bias[n];
    if (a.col_scale) t.scale = a.col_scale[n];
    if (a.residual) t.residual = a.residual[(int64_t)m * a.ldc + n];
  }
  return t;
}
__device__ __forceinline__ float first_output(const GemmArgs& a, const PutTerms& t, float acc) {
  float v = fmaf(acc, a.alpha, t.bias);
  if (a.col_scale) v *= t.scale;
  if (a.residual) v += t.residual;
  return v;
}
__device__ __forceinline__ void put_second(const GemmArgs& a, int m, int n, float acc) {
  put_c2(a, (int64_t)m * a.ldc2 + (n - a.n_first), dh::activate(acc * a.alpha, a.act));
}

// Where a workgroup's tile lies: its rows (base + 0 .. rows - 1 of the outputs), its first row among them, its weights.
struct TilePlace {
  int base, rows, m0;
  const uint16_t* W;
};
template <bool GROUPED>
__device__ __forceinline__ bool place_tile(const GemmArgs& a, int m_tile, int bm, TilePlace* p) {
  p->base = 0; p->rows = a.M; p->m0 = m_tile * bm; p->W = a.W;
  if (GROUPED) {
    const int g = a.rows.tiles[2 * m_tile];
    if (g < 0) return false;
    p->m0 = a.rows.tiles[2 * m_tile + 1];
    p->base = a.rows.group_off[g];
    p->rows = a.rows.group_off[g + 1] - p->base;
    p->W += (int64_t)g * a.rows.w_stride;
  }
  return true;
}
// The activation row behind a tile's row (rows past the group repeat its last one: their products are never stored).
template <bool GROUPED>
__device__ __forceinline__ int64_t source_row(const GemmArgs& a, const TilePlace& p, int row) {
  const int r = p.base + min(p.m0 + row, p.rows - 1);
  return GROUPED && a.rows.row_index ? a.rows.row_index[r] : r;
}

// One 32 x 32 accumulator tile: lane l holds column l & 31 and rows 8 (i / 4) + 4 (l >> 5) + i % 4.
//
// An epilogue requests all it adds and multiplies in (several tiles' residuals at a time) in front of its first store, and computes a tile's
// values before it stores them: a load behind a store waits for the store's trip to memory as well, and values between the branches of
// ragged rows are computed one after the other.  Sixteen round trips for a tile of gated pairs took 18 us of 68 (1531 x 6144 x 2048).
// A small product waits for every instruction of it, so kernels with and without a residual are two, addresses are a multiplication of 32
// bits a row, fours of rows that a tile does not have are left out, raw sums of k slices are one kernel's, and first and second outputs follow one
// another: settled at every value, each steps over the other's code (us, one form and sixteen rows for all -> now: 40 x 1024 x 1024 6.96 -> 6.6, 4 x 119 x 192
// with the exact gelu 4.36 -> 3.65, 500 x 500 x 448 with a residual 5.36 -> 5.3, 996 x 3600 x 1472 with both outputs 34.1 -> 27.5).
__device__ __forceinline__ int tile_row(int mb, int i) { return mb + 8 * (i >> 2) + (i & 3); }

struct ColumnTerms {       // of one column of the first output
  float alpha, bias;
};
__device__ __forceinline__ ColumnTerms column_terms(const GemmArgs& a, int n0, int lane) {
  const int n = min(n0 + (lane & 31), a.n_first - 1);
  const float bias = a.bias ? a.bias[n] : 0.f, scale = a.col_scale ? a.col_scale[n] : 1.f;
  return {a.alpha * scale, bias * scale};
}
// (every read in front of the first write, also because the residual may be the output itself)
__device__ __forceinline__ void load_residual(const GemmArgs& a, const TilePlace& p, float (&r)[16], int m0, int n0, int lane) {
  const int n = n0 + (lane & 31), mb = m0 + 4 * (lane >> 5);
  const float* res = a.residual + (int64_t)p.base * a.ldc + min(n, a.n_first - 1);
#pragma unroll
  for (int i = 0; i < 16; i++) r[i] = res[(int64_t)min(tile_row(mb, i), p.rows - 1) * a.ldc];
}
// value(i) for the fours of rows that a wave's tile at m0 has.
template <class Value>
__device__ __forceinline__ void by_fours(int m0, int rows, Value&& value) {
#pragma unroll
  for (int q = 0; q < 4; q++)
    if (m0 + 8 * q < rows)
#pragma unroll
      for (int i = 4 * q; i < 4 * q + 4; i++) value(i);
}
template <class T, class Value>
__device__ __forceinline__ void store_rows(T* c, int ld, int mb, int rows, Value&& value) {
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int m = tile_row(mb, i);
    if (m < rows) c[(int64_t)m * ld] = value(i);
  }
}
__device__ __forceinline__ void store_c2(const GemmArgs& a, int64_t at, int mb, int rows, const float (&v)[16]) {
  if (a.c2_dtype == DH_BF16) store_rows(static_cast<uint16_t*>(a.C2) + at, a.ldc2, mb, rows, [&](int i) { return dh::f32_to_bf16_bits(v[i]); });
  else if (a.c2_dtype == DH_F16) store_rows(static_cast<_Float16*>(a.C2) + at, a.ldc2, mb, rows, [&](int i) { return (_Float16)v[i]; });
  else store_rows(static_cast<float*>(a.C2) + at, a.ldc2, mb, rows, [&](int i) { return v[i]; });
}
template <class Flag>
__device__ __forceinline__ void store_first(const GemmArgs& a, const TilePlace& p, const f32x16_t& acc, const ColumnTerms& col, Flag with_residual,
                                            const float (&r)[16], int m0, int n0, int lane) {
  const int n = n0 + (lane & 31), mb = m0 + 4 * (lane >> 5);
  if (n >= a.n_first) return;
  float* c = a.C + (int64_t)p.base * a.ldc + n;
  if (with_residual) store_rows(c, a.ldc, mb, p.rows, [&](int i) { return fmaf(acc[i], col.alpha, col.bias) + r[i]; });
  else store_rows(c, a.ldc, mb, p.rows, [&](int i) { return fmaf(acc[i], col.alpha, col.bias); });
}
template <int ACT, bool FEW>
__device__ __forceinline__ void store_second(const GemmArgs& a, const TilePlace& p, const f32x16_t& acc, int m0, int n0, int lane) {
  const int n = n0 + (lane & 31), mb = m0 + 4 * (lane >> 5);
  if (n < a.n_first || n >= a.N) return;
  const int64_t at = (int64_t)p.base * a.ldc2 + (n - a.n_first);
  if (ACT == kAnyAct || (FEW && m0 + 8 >= p.rows)) {      // one value at a time: sixteen of each activation are too much code, and few rows have few values
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int m = tile_row(mb, i);
      if (m < p.rows) put_c2(a, at + (int64_t)m * a.ldc2, dh::activate(acc[i] * a.alpha, ACT == kAnyAct ? a.act : ACT));
    }
  } else {
    float v[16];
    by_fours(m0, p.rows, [&](int i) { v[i] = dh::activate(acc[i] * a.alpha, ACT); });
    store_c2(a, at, mb, p.rows, v);
  }
}
// First outputs of tiles AT .. of a wave's R x C; residuals of four tiles at a time.
template <int AT, int R, int C, class Flag>
__device__ __forceinline__ void store_from(const GemmArgs& a, const TilePlace& p, const f32x16_t (&acc)[R][C], const ColumnTerms (&col)[C],
                                           Flag with_residual, int m0, int n0, int lane) {
  constexpr int kBatch = R * C < 4 ? R * C : 4;
  float r[kBatch][16];
  if (with_residual) {
#pragma unroll
    for (int u = 0; u < kBatch; u++) load_residual(a, p, r[u], m0 + 32 * ((AT + u) / C), n0 + 32 * ((AT + u) % C), lane);
  }
#pragma unroll
  for (int u = 0; u < kBatch; u++)
    store_first(a, p, acc[(AT + u) / C][(AT + u) % C], col[(AT + u) % C], with_residual, r[u], m0 + 32 * ((AT + u) / C), n0 + 32 * ((AT + u) % C), lane);
  if constexpr (AT + kBatch < R * C) store_from<AT + kBatch>(a, p, acc, col, with_residual, m0, n0, lane);
}
// A wave's tiles: raw sums of a k slice (kernels that are launched with slices), or first outputs and then second ones.
template <int ACT, bool SLICES, int R, int C>
__device__ __forceinline__ void store_tiles(const GemmArgs& a, const TilePlace& p, const f32x16_t (&acc)[R][C], int m0, int n0, int lane) {
  if (SLICES && a.parts) {
#pragma unroll
    for (int t = 0; t < R * C; t++) {
      const int n = n0 + 32 * (t % C) + (lane & 31);
      if (n < a.N) store_rows(a.parts + (int64_t)blockIdx.y * a.M * a.N + n, a.N, m0 + 32 * (t / C) + 4 * (lane >> 5), a.M, [&](int i) { return acc[t / C][t % C][i]; });
    }
    return;
  }
  if (n0 < a.n_first) {
    ColumnTerms col[C];
#pragma unroll
    for (int j = 0; j < C; j++) col[j] = column_terms(a, n0 + 32 * j, lane);
    if constexpr (ACT == kNoSecond) store_from<0>(a, p, acc, col, std::false_type{}, m0, n0, lane);
    else if constexpr (R * C > 4) store_from<0>(a, p, acc, col, a.residual != nullptr, m0, n0, lane);    // (known, registers are spilled here)
    else if (ACT == kResidual || a.residual) store_from<0>(a, p, acc, col, std::true_type{}, m0, n0, lane);
    else store_from<0>(a, p, acc, col, std::false_type{}, m0, n0, lane);
  }
  if constexpr (!only_first(ACT)) {
    if (n0 + 32 * C > a.n_first)
#pragma unroll
      for (int t = 0; t < R * C; t++) store_second<ACT, R * C == 1>(a, p, acc[t / C][t % C], m0 + 32 * (t / C), n0 + 32 * (t % C), lane);
  }
}
// The same for R gate tiles and the up tiles beside them (first weight row n0 of the gate block).
template <int R>
__device__ __forceinline__ void store_glu(const GemmArgs& a, const TilePlace& p, const f32x16_t (&acc)[R][2], int m0, int n0, int lane) {
  if (n0 >= a.N) return;
  const int mb = m0 + 4 * (lane >> 5);
  float f[R][16];          // a row's factor, on what goes in or on what comes out
  if (a.rows.factor) {
#pragma unroll
    for (int t = 0; t < R; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) f[t][i] = a.rows.factor[p.base + min(tile_row(mb + 32 * t, i), p.rows - 1)];
  } else {
#pragma unroll
    for (int t = 0; t < R; t++)
#pragma unroll
      for (int i = 0; i < 16; i++) f[t][i] = 1.f;
  }
  const bool in = a.rows.factor_in;
#pragma unroll
  for (int t = 0; t < R; t++) {
    float y[16];
    by_fours(m0 + 32 * t, p.rows, [&](int i) {
      const float w = in ? f[t][i] : 1.f;
      y[i] = dh::clamped_glu(w * acc[t][0][i], w * acc[t][1][i], a.rows.limit) * (in ? 1.f : f[t][i]);
    });
    store_c2(a, (int64_t)p.base * a.ldc2 + (n0 >> 1) + (lane & 31), mb + 32 * t, p.rows, y);
  }
}

// 16-bit operands (gemm_wide.h): the tile of workgroup `block`.
template <class Tile, bool F16, int ACT, bool GROUPED, bool GLU>
__device__ __forceinline__ void gemm_16bit(const GemmArgs& a, int block, char* smem) {
  static_assert(!GLU || Tile::FB == 1 || Tile::FA == 0, "a wave's two tiles are the gate and the up value");
  const int tile = dh::xcd_contiguous(block, a.tiles_m * a.tiles_n);
  TilePlace place;
  if (!place_tile<GROUPED>(a, tile % a.tiles_m, Tile::BM, &place)) return;
  const int m0 = place.m0, n0 = (tile / a.tiles_m) * Tile::BN;
  const int k0 = blockIdx.y * a.k_slice, nk = min(a.k_slice, a.K - k0) >> 6;
  // offsets count from the tile's first row, which may lie anywhere; those of gathered rows from the first of all
  const int64_t first = GROUPED && a.rows.row_index ? 0 : (int64_t)place.base + m0;
  const void *a_base = static_cast<const uint16_t*>(a.A) + first * a.lda, *w_base = place.W + (int64_t)n0 * a.ldw;
  auto a_off = [&](int row) { return (uint32_t)((source_row<GROUPED>(a, place, row) - first) * a.lda * 2); };
  auto w_off = [&](int row) { return (uint32_t)(min(row, a.N - 1 - n0) * a.ldw * 2); };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave / Tile::WN, wn = wave % Tile::WN;
  const dh::Company company{m0 / Tile::BM, (place.rows + Tile::BM - 1) / Tile::BM};
  if constexpr (Tile::FA == 0) {
    f32x16_t acc[1][Tile::G];
    dh::small_product<Tile, F16>(acc[0], a_base, a_off, w_base, w_off, 2u * k0, nk, smem, company);
    const int m = m0 + 32 * wm, n = n0 + 32 * Tile::G * wn;
    if constexpr (GLU) store_glu(a, place, acc, m, n, lane);
    else store_tiles<ACT, ACT == kNoSecond && !GROUPED>(a, place, acc, m, n, lane);
  } else {
    f32x16_t acc[2 * Tile::FA][2 * Tile::FB];
    dh::wide_product<Tile, F16>(acc, a_base, a_off, w_base, w_off, 2u * k0, nk, smem, company);
    const int m = m0 + 64 * Tile::FA * wm, n = n0 + 64 * Tile::FB * wn;
    if constexpr (GLU) store_glu(a, place, acc, m, n, lane);
    else store_tiles<ACT, ACT == kNoSecond && !GROUPED>(a, place, acc, m, n, lane);
  }
}

template <class Tile, bool F16, int ACT, bool GROUPED = false, bool GLU = false>
__global__ __launch_bounds__(Tile::kThreads, 2) void gemm_16bit_kernel(const GemmArgs a) {
  extern __shared__ __align__(16) char smem[];
  gemm_16bit<Tile, F16, ACT, GROUPED, GLU>(a, blockIdx.x, smem);
}
// A shared expert's product and the routed experts' beside it: own_blocks (a multiple of eight, so that both find their dies) for the first.
template <class Tile, bool GLU>
__global__ __launch_bounds__(Tile::kThreads, 2) void gemm_experts_kernel(const GemmArgs shared, const GemmArgs routed, int own_blocks) {
  extern __shared__ __align__(16) char smem[];
  const int block = blockIdx.x;
  if (block >= own_blocks) gemm_16bit<Tile, false, kNoSecond, true, GLU>(routed, block - own_blocks, smem);
  else if (block < shared.tiles_m * shared.tiles_n) gemm_16bit<Tile, false, kNoSecond, false, GLU>(shared, block, smem);
}

// The 32-bit product: four waves, a 64 x 64 TN tile, 32 k at a time.  Both tiles sit in LDS as f32 rows of 32 + 4
// words; a lane reads four consecutive k of its row and feeds four instructions with them (k-slot l >> 5 of
// instruction e stands for k = 8 s + 4 (l >> 5) + e on both sides).  A matrix-core instruction takes 64 cycles here, so a tile's 16
// of them cover the loads of the next (registers, then the other LDS buffer; one barrier a tile).  k slices (blockIdx.y) as for the
// 16-bit ones.
template <int TN, bool GROUPED, bool GLU>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const GemmArgs a) {
  static_assert(!GLU || TN == 2, "a wave's two tiles are the gate and the up value");
  constexpr int BM = 64, BN = 64 * TN, BK = 32, ROW = BK + 4;
  __shared__ __align__(16) float la[2][BM * ROW];
  __shared__ __align__(16) float lb[2][BN * ROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int tile = dh::xcd_contiguous(blockIdx.x, a.tiles_m * a.tiles_n);
  TilePlace place;
  if (!place_tile<GROUPED>(a, tile % a.tiles_m, BM, &place)) return;
  const int m0 = place.m0, n0 = (tile / a.tiles_m) * BN;
  const int k0 = blockIdx.y * a.k_slice, nk = min(a.k_slice, a.K - k0) / BK;
  // A: 64 rows x 8 pieces of 4 floats, two per thread; W: 64 TN rows x 4 pieces of 8 elements, TN per thread
  const float* pa[2];
  const uint16_t* pb[TN];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int p = tid + 256 * r;
    pa[r] = static_cast<const float*>(a.A) + source_row<GROUPED>(a, place, p >> 3) * a.lda + 4 * (p & 7) + k0;
  }
#pragma unroll
  for (int r = 0; r < TN; r++) pb[r] = place.W + (int64_t)min(n0 + 64 * r + (tid >> 2), a.N - 1) * a.ldw + 8 * (tid & 3) + k0;
  f32x4_t ra[2];
  u32x4_t rb[TN];
  f32x16_t acc[1][TN];
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[0][j][e] = 0.f;
  auto load = [&](int kt) {
#pragma unroll
    for (int r = 0; r < 2; r++) ra[r] = *reinterpret_cast<const f32x4_t*>(pa[r] + BK * kt);
#pragma unroll
    for (int r = 0; r < TN; r++) rb[r] = *reinterpret_cast<const u32x4_t*>(pb[r] + BK * kt);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const int p = tid + 256 * r;
      *reinterpret_cast<f32x4_t*>(&la[buf][(p >> 3) * ROW + 4 * (p & 7)]) = ra[r];
    }
#pragma unroll
    for (int r = 0; r < TN; r++) {
      f32x4_t* wb = reinterpret_cast<f32x4_t*>(&lb[buf][(64 * r + (tid >> 2)) * ROW + 8 * (tid & 3)]);
      wb[0] = f32x4_t{dh::bf16_low(rb[r][0]), dh::bf16_high(rb[r][0]), dh::bf16_low(rb[r][1]), dh::bf16_high(rb[r][1])};
      wb[1] = f32x4_t{dh::bf16_low(rb[r][2]), dh::bf16_high(rb[r][2]), dh::bf16_low(rb[r][3]), dh::bf16_high(rb[r][3])};
    }
  };
  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < nk; kt++) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load(kt + 1);
#pragma unroll
    for (int s = 0; s < BK / 8; s++) {
      const int k = 8 * s + 4 * (lane >> 5);
      const f32x4_t fa = *reinterpret_cast<const f32x4_t*>(&la[buf][(32 * wm + (lane & 31)) * ROW + k]);
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const f32x4_t fb = *reinterpret_cast<const f32x4_t*>(&lb[buf][(32 * (wn * TN + j) + (lane & 31)) * ROW + k]);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc[0][j], 0, 0, 0);
      }
    }
    if (kt + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }
  if constexpr (GLU) store_glu(a, place, acc, m0 + 32 * wm, n0 + 32 * wn * TN, lane);
  else store_tiles<kAnyAct, !GROUPED>(a, place, acc, m0 + 32 * wm, n0 + 32 * wn * TN, lane);
}

// 32-bit products of rows within reach (gemm_split.h).  Bound by the matrix cores where tiles are many (at 600 x 18464 x 4096 the three
// instructions' rate is 1060 TFLOP/s, what the 16-bit products reach), by the steps' latency where they are few; us against 32-bit
// instructions: 301 x 5136 x 1024 43 -> 18, 301 x 1024 x 4096 37 -> 18, 600 x 18464 x 4096 893 -> 257, 2 x 4096 x 16384 83 -> 34.
// Distance from 64 bits (2-norm) there 5.7e-7 -> 1.0e-7, 4.7e-7 -> 1.4e-7, 8.1e-7 -> 2.7e-7, 8.1e-7 -> 2.2e-7.  A tile with sums the parts do not
// give (an activation that is not the sum of its parts, sound_sum) is multiplied again by 32-bit instructions, and those sums are taken from there.
template <class Tile>
__global__ __launch_bounds__(Tile::kThreads, Tile::kPerSimd) void gemm_split_kernel(const GemmArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int tile = dh::xcd_contiguous(blockIdx.x, a.tiles_m * a.tiles_n);
  TilePlace place;
  place_tile<false>(a, tile % a.tiles_m, Tile::BM, &place);
  const int m0 = place.m0, n0 = (tile / a.tiles_m) * Tile::BN;
  const int k0 = blockIdx.y * a.k_slice, k_end = min(k0 + a.k_slice, a.K);
  const float* a_base = static_cast<const float*>(a.A) + (int64_t)m0 * a.lda + k0;
  const uint16_t* w_base = a.W + (int64_t)n0 * a.ldw + k0;
  auto a_off = [&](int row) { return (uint32_t)((int64_t)min(row, a.M - 1 - m0) * a.lda * 4); };
  auto w_off = [&](int row) { return (uint32_t)((int64_t)min(row, a.N - 1 - n0) * a.ldw * 2); };
  const int nk = (k_end - k0) >> 6;
  dh::f32x4_t sums[Tile::kShare];
  const bool whole = dh::split_product<Tile>(a_base, a_off, w_base, w_off, nk, smem), sound = dh::join_sums<Tile>(sums, smem);
  if (__builtin_expect(!dh::everywhere<Tile>(whole && sound, smem), 0)) {
    const int* const short_rows = dh::short_rows<Tile>(whole, smem);
    dh::exact_product<Tile>(a_base, a_off, w_base, w_off, nk, smem);
    __syncthreads();
    dh::f32x4_t exact[Tile::kShare];
    (void)dh::join_sums<Tile>(exact, smem);
    // (the other sums stay what they are whatever the rest of their tile holds)
#pragma unroll
    for (int u = 0; u < Tile::kShare; u++) {
      const dh::SumPlace<Tile> at(u);
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (short_rows[32 * at.wm + 8 * at.q + 4 * ((threadIdx.x & 63) >> 5) + e] || !dh::sound_sum(sums[u][e])) sums[u][e] = exact[u][e];
    }
  }
  const int lane = threadIdx.x & 63;
  // (which output a tile has is settled in front of the loops over its sums: stepping over the other's code at each of them took 0.7 us)
  auto each = [&](auto&& f) {
#pragma unroll
    for (int u = 0; u < Tile::kShare; u++) {
      const dh::SumPlace<Tile> at(u);
      const int n = n0 + 32 * at.j + (lane & 31), m = m0 + 32 * at.wm + 8 * at.q + 4 * (lane >> 5);
#pragma unroll
      for (int e = 0; e < 4; e++) f(u, e, m + e, n);
    }
  };
  if (a.parts) {
    each([&](int u, int e, int m, int n) {
      if (m < a.M && n < a.N) a.parts[((int64_t)blockIdx.y * a.M + m) * a.N + n] = sums[u][e];
    });
    return;
  }
  if (n0 < a.n_first) {
    if (has_terms(a)) {
      PutTerms terms[Tile::kShare][4];
      each([&](int u, int e, int m, int n) { terms[u][e] = put_terms(a, min(m, a.M - 1), n); });
      each([&](int u, int e, int m, int n) {
        if (m < a.M && n < a.n_first) a.C[(int64_t)m * a.ldc + n] = first_output(a, terms[u][e], sums[u][e]);
      });
    } else {
      each([&](int u, int e, int m, int n) {
        if (m < a.M && n < a.n_first) a.C[(int64_t)m * a.ldc + n] = fmaf(sums[u][e], a.alpha, 0.f);
      });
    }
  }
  if (n0 + Tile::BN > a.n_first)
    each([&](int u, int e, int m, int n) {
      if (m < a.M && n >= a.n_first && n < a.N) put_second(a, m, n, sums[u][e]);
    });
}

// Sums of the k slices in slice order.  VEC columns per thread (N a multiple of VEC), a block's threads as wide as the row allows and the
// rest of them on further rows (thread t: column t % wide, row t / wide); a grid's second dimension holds 65535 blocks, so rows go round.
template <int VEC>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmArgs a, int slices, int log2_wide, int round) {
  const int n = VEC * ((blockIdx.x << log2_wide) + (threadIdx.x & ((1 << log2_wide) - 1)));
  if (n >= a.N) return;
  const int64_t total = (int64_t)a.M * a.N;
  for (int m = (blockIdx.y << (8 - log2_wide)) + (threadIdx.x >> log2_wide); m < a.M; m += round) {
    const float* p = a.parts + (int64_t)m * a.N + n;
    float s[VEC] = {};
    PutTerms terms[VEC];
    const bool whole = VEC == 4 && n + 3 < a.n_first && a.ldc % 4 == 0 && ((reinterpret_cast<uintptr_t>(a.C) | reinterpret_cast<uintptr_t>(a.residual)) & 15) == 0;
    const bool with_terms = has_terms(a) && n < a.n_first;
    if (with_terms) {
      f32x4_t residual = {0.f, 0.f, 0.f, 0.f};
      if (whole && a.residual) residual = *reinterpret_cast<const f32x4_t*>(a.residual + (int64_t)m * a.ldc + n);
#pragma unroll
      for (int e = 0; e < VEC; e++) {
        if (whole) terms[e] = PutTerms{a.bias ? a.bias[n + e] : 0.f, a.col_scale ? a.col_scale[n + e] : 1.f, residual[e]};
        else terms[e] = put_terms(a, m, n + e);
      }
    }
#pragma unroll 4
    for (int k = 0; k < slices; k++) {
      if constexpr (VEC == 4) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(p + k * total);
#pragma unroll
        for (int e = 0; e < 4; e++) s[e] += v[e];
      } else {
        s[0] += p[k * total];
      }
    }
    float v[VEC];
#pragma unroll
    for (int e = 0; e < VEC; e++) v[e] = with_terms ? first_output(a, terms[e], s[e]) : fmaf(s[e], a.alpha, 0.f);
    if (whole) {
      *reinterpret_cast<f32x4_t*>(a.C + (int64_t)m * a.ldc + n) = f32x4_t{v[0], v[VEC > 1 ? 1 : 0], v[VEC > 2 ? 2 : 0], v[VEC > 3 ? 3 : 0]};
    } else {
#pragma unroll
      for (int e = 0; e < VEC; e++) {
        if (n + e < a.n_first) a.C[(int64_t)m * a.ldc + n + e] = v[e];
        else put_second(a, m, n + e, s[e]);
      }
    }
  }
}

// The same where all columns are a first output's and the rows are normed behind it: one workgroup a row (N a multiple of 4, at most 4096, everything
// aligned).  The norm's launch was 3.1 us and 1.4 in front of the next: 301 rows of 1024 in three slices 4.4 + 3.1 -> 5.0 us.
template <bool BF16>
__global__ __launch_bounds__(256) void gemm_reduce_norm_kernel(const GemmArgs a, int slices) {
  __shared__ float red[4];
  const int m = blockIdx.x;
  const int64_t total = (int64_t)a.M * a.N;
  const float *p = a.parts + (int64_t)m * a.N, *res = a.residual ? a.residual + (int64_t)m * a.ldc : nullptr;
  float* c = a.C + (int64_t)m * a.ldc;
  float4 x[dh::kMadePieces];
#pragma unroll
  for (int j = 0; j < dh::kMadePieces; j++) {
    const int n = 4 * (threadIdx.x + 256 * j);
    x[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (n >= a.N) continue;
    f32x4_t bias = {0.f, 0.f, 0.f, 0.f}, scale = {1.f, 1.f, 1.f, 1.f}, residual = bias, s = bias;
    if (a.bias) bias = *reinterpret_cast<const f32x4_t*>(a.bias + n);
    if (a.col_scale) scale = *reinterpret_cast<const f32x4_t*>(a.col_scale + n);
    if (res) residual = *reinterpret_cast<const f32x4_t*>(res + n);
#pragma unroll 4
    for (int k = 0; k < slices; k++) s += *reinterpret_cast<const f32x4_t*>(p + k * total + n);
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = first_output(a, PutTerms{bias[e], scale[e], residual[e]}, s[e]);
    x[j] = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(c + n) = x[j];
  }
  dh::store_normed_row<BF16>(x, a.N, a.norm_weight, a.norm_eps, red, a.normed, (int64_t)m * a.ld_normed, a.ld_normed);
}

// Tiles of the 16-bit products, and what they cost in ns: a k step (64 elements) `alone` with few workgroups on the device, `one` with one
// on every compute unit, `full` with as many as fit (the two larger tiles: one, which takes more than half of the LDS); outside the k
// loop `start`, and `again` for every further round of workgroups.  The device slows its clock under matrix-core load, so a step gets
// dearer as more compute units join, and idle ones are not all lost.  Fitted to 300 products (M 16 .. 2100, N 200 .. 20000, K 256 .. 16384) with each
// tile and up to 16 slices, weights from HBM as a model's layers in turn have them: the choice is 0.5 % behind the best on average, 15 % at
// worst (1.1 % and 30 % with the costs of tiles that did not ask for their weights ahead).
// Against the 128 x 128 and 64 x 64 tiles through registers that were here before, us: 2048 x 18464 x 4096
// 421 -> 299, 2048 x 4096 x 16384 329 -> 224, 1531 x 2048 x 6144 70 -> 51, 300 x 2048 x 2048 18.4 -> 11.3, 33 x 5120 x 1024 14.6 -> 7.2,
// 700 x 1024 x 1024 14.1 -> 7.4; behind them still: 33 x 4096 x 16384 30.6 -> 33.1 (2 rows 28.5 -> 32.7) and few rows at K 64.
using Tile256x256 = dh::WideTile<2, 4, 2, 1>;
using Tile256x128 = dh::WideTile<4, 2, 1, 1>;
using Tile128x128 = dh::WideTile<2, 2, 1, 1>;
using Tile64x64 = dh::SmallTile<2, 2, 1>;
using Tile64x128 = dh::SmallTile<2, 2, 2>;     // gate and up columns
struct TileCost {
  int bm, bn, per_cu;
  float alone, one, full, start, again;
};
constexpr TileCost kTiles[] = {{256, 256, 1, 993.f, 1464.f, 1627.f, 8987.f, 8447.f},
                               {256, 128, 1, 457.f, 808.f, 899.f, 11078.f, 4801.f},
                               {128, 128, 2, 396.f, 619.f, 1337.f, 5092.f, 2173.f},
                               {64, 64, 2, 163.f, 294.f, 498.f, 5060.f, 803.f}};
// gate and up products, never sliced (costs of tiles that did not ask for their weights ahead, not fitted again since)
constexpr TileCost kGluTiles[] = {{256, 256, 1, 900.f, 1720.f, 1720.f, 8000.f, 0.f},
                                  {256, 128, 1, 520.f, 930.f, 930.f, 5500.f, 0.f},
                                  {128, 128, 2, 330.f, 480.f, 1080.f, 4500.f, 0.f},
                                  {64, 128, 1, 260.f, 330.f, 330.f, 3700.f, 0.f}};
constexpr int kMaxSlices = 16, kMinSliceSteps = 8;

struct TileChoice {
  int tile, slices;
  double ns = 0.0;
};
// The k loops of so many workgroups; `lone`: how much of the full step's time a single workgroup on every compute unit would take.
double loops_ns(const TileCost& c, int64_t groups, int64_t steps, double lone) {
  const int64_t cus = dh::num_cus(), slots = cus * c.per_cu, left = groups % slots;
  const double f = (double)left / cus;
  const double step = f <= 1.0 ? c.alone + (c.one - c.alone) * f : c.full * (lone + (1.0 - lone) * f / c.per_cu);
  const int64_t rounds = groups / slots + (left ? 1 : 0);
  return steps * ((double)(groups / slots) * c.full + (left ? step : 0.0)) + (double)(rounds - 1) * c.again;
}
// The cheapest tile and number of k slices.  Slices cost the round trip of their raw sums (about 4 TB/s) and a second launch, and no
// number of them is faster than the weights come in.
// erf: a second output through the exact gelu, whose epilogue takes a compute unit about 60 ns for each element a lane holds of a wave, 40
// where another workgroup's loop runs beside it (1531 x 6144 x 2048 without it 52 us on 128 x 128 tiles, 47 on 256 x 256; with it 76 and
// 111); behind slices it is the reduce launch's.
TileChoice choose_tile(int64_t M, int64_t N, int64_t K, int most_slices, bool glu, bool erf) {
  const int64_t steps = K / 64;
  TileChoice best{0, 1};
  double least = 1e30;
  for (int i = 0; i < 4; i++) {
    const TileCost& c = glu ? kGluTiles[i] : kTiles[i];
    for (int s = 1; s <= most_slices && (s == 1 || steps / s >= kMinSliceSteps); s++) {
      const int64_t groups = dh::ceil_div(M, c.bm) * dh::ceil_div(N, c.bn) * s;
      double t = std::max(loops_ns(c, groups, dh::ceil_div(steps, s), 0.76), 2.0 * N * K / (glu ? 6450.0 : 6950.0)) + c.start;
      if (s > 1) t += 2550.0 + 4.0 * M * N * (2 * s + 1) / 4300.0;
      else if (erf) t += (c.per_cu == 1 ? 60.0 : 40.0) * (c.bm * c.bn / 64) * dh::ceil_div(groups, dh::num_cus());
      if (t < least) {
        least = t;
        best = TileChoice{i, s, t};
      }
    }
  }
  return best;
}

// A tile's rows are addressed by 32-bit byte offsets from its first (rows millions of elements long are out of reach; a single row never is).
bool within_reach(int64_t rows, int64_t ld, int64_t K) { return 2 * ((std::min<int64_t>(rows, 256) - 1) * ld + K) < (int64_t)1 << 32; }

// k of a slice (whole steps of 64).
int slice_extent(int64_t K, int slices) { return (int)dh::ceil_div(K / 64, slices) * 64; }

// LDS beyond 64 KB is asked for once per kernel.
template <class Tile, bool F16, int ACT, bool GROUPED, bool GLU>
int launch_16bit_kernel(const char* op, GemmArgs a, int slices) {
  auto kern = gemm_16bit_kernel<Tile, F16, ACT, GROUPED, GLU>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::kLds);
  DH_CHECK_HIP(op, set);
  const bool gathered = GROUPED && a.rows.row_index;
  if (!(gathered ? (int64_t)2 * a.rows.source_rows * a.lda < (int64_t)1 << 32 : within_reach(GROUPED ? Tile::BM : a.M, a.lda, a.K)) || !within_reach(a.N, a.ldw, a.K))
    return dh::fail(1, "[%s] rows %lld and %lld elements apart are out of reach", op, (long long)a.lda, (long long)a.ldw);
  if (!GROUPED) a.tiles_m = (int)dh::ceil_div(a.M, Tile::BM);
  a.tiles_n = (int)dh::ceil_div(a.N, Tile::BN);
  hipLaunchKernelGGL(kern, dim3(a.tiles_m * a.tiles_n, slices), dim3(Tile::kThreads), Tile::kLds, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}
int launch_reduce(const char* op, const GemmArgs& a, int slices) {
  if (a.norm_weight && a.n_first == a.N && a.N % 4 == 0 && a.N <= 1024 * dh::kMadePieces && a.ldc % 4 == 0 &&
      ((reinterpret_cast<uintptr_t>(a.C) | reinterpret_cast<uintptr_t>(a.residual) | reinterpret_cast<uintptr_t>(a.bias) |
        reinterpret_cast<uintptr_t>(a.col_scale)) & 15) == 0) {
    auto kern = a.normed_dtype == DH_BF16 ? gemm_reduce_norm_kernel<true> : gemm_reduce_norm_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(a.M), dim3(256), 0, dh::stream(), a, slices);
    DH_CHECK_LAUNCH(op);
    *a.norm_done = true;
    return 0;
  }
  const bool vec = a.N % 4 == 0;
  const int64_t columns = vec ? a.N / 4 : a.N;
  int log2_wide = 8;
  while (log2_wide > 2 && 1 << (log2_wide - 1) >= columns) log2_wide--;
  const int rows = 256 >> log2_wide;
  const dim3 grid((unsigned)dh::ceil_div(columns, 1 << log2_wide), (unsigned)std::min<int64_t>(dh::ceil_div(a.M, rows), 65535));
  if (vec) hipLaunchKernelGGL(gemm_reduce_kernel<4>, grid, dim3(256), 0, dh::stream(), a, slices, log2_wide, rows * (int)grid.y);
  else hipLaunchKernelGGL(gemm_reduce_kernel<1>, grid, dim3(256), 0, dh::stream(), a, slices, log2_wide, rows * (int)grid.y);
  DH_CHECK_LAUNCH(op);
  return 0;
}
template <bool F16, int ACT, bool GLU>
int launch_16bit(const char* op, GemmArgs a, const TileChoice& pick) {
  a.k_slice = a.K;
  int slices = 1;
  if (pick.slices > 1) {
    a.k_slice = (int)dh::ceil_div(a.K / 64, pick.slices) * 64;
    slices = (int)dh::ceil_div(a.K, a.k_slice);
    size_t bytes = 0;
    a.parts = dh::splitk_workspace(&bytes);
  }
  int rc;
  switch (pick.tile) {
    case 0: rc = launch_16bit_kernel<Tile256x256, F16, ACT, false, GLU>(op, a, slices); break;
    case 1: rc = launch_16bit_kernel<Tile256x128, F16, ACT, false, GLU>(op, a, slices); break;
    case 2: rc = launch_16bit_kernel<Tile128x128, F16, ACT, false, GLU>(op, a, slices); break;
    default: rc = launch_16bit_kernel<std::conditional_t<GLU, Tile64x128, Tile64x64>, F16, ACT, false, GLU>(op, a, slices); break;
  }
  if (rc || !a.parts) return rc;
  return launch_reduce(op, a, slices);
}
int launch_act(const char* op, const GemmArgs& a, bool f16, const TileChoice& pick) {
  // (behind slices terms and second outputs are the reduce launch's)
  if (a.K > slice_extent(a.K, pick.slices) || (a.n_first == a.N && !a.residual))
    return f16 ? launch_16bit<true, kNoSecond, false>(op, a, pick) : launch_16bit<false, kNoSecond, false>(op, a, pick);
  if (f16) return a.n_first == a.N ? launch_16bit<true, kResidual, false>(op, a, pick)
                  : a.act == DH_ACT_NONE ? launch_16bit<true, DH_ACT_NONE, false>(op, a, pick)
                                         : launch_16bit<true, kAnyAct, false>(op, a, pick);
  if (a.n_first == a.N) return launch_16bit<false, kResidual, false>(op, a, pick);
  if (a.act == DH_ACT_RELU2) return launch_16bit<false, DH_ACT_RELU2, false>(op, a, pick);
  if (a.act == DH_ACT_GELU_ERF) return launch_16bit<false, DH_ACT_GELU_ERF, false>(op, a, pick);
  return launch_16bit<false, kAnyAct, false>(op, a, pick);
}

// k slices that the library's workspace holds the sums of.
int slices_in_workspace(int64_t M, int64_t N, int most) {
  size_t ws_bytes = 0;
  (void)dh::splitk_workspace(&ws_bytes);
  return (int)std::max<size_t>(1, std::min<size_t>(most, ws_bytes / ((size_t)M * N * sizeof(float))));
}
TileChoice choose_16bit(int64_t M, int64_t N, int64_t K, bool erf) {
  const int most = slices_in_workspace(M, N, kMaxSlices);
  TileChoice pick = choose_tile(M, N, K, most, false, erf);
  const int env_tile = dh::tuning_int("DH_DENSE_TILE", -1), env_slices = dh::tuning_int("DH_DENSE_SLICES", 0);
  if (env_tile >= 0) pick.tile = env_tile;
  if (env_slices) pick.slices = std::min(most, env_slices);
  return pick;
}

// A product whose rows are out of reach goes in halves.
int dense_16bit(const char* op, const GemmArgs& whole, bool f16) {
  GemmArgs a = whole;
  if ((a.M > 1 && !within_reach(a.M, a.lda, a.K)) || (a.N > 1 && !within_reach(a.N, a.ldw, a.K))) a.norm_weight = nullptr;      // (its rows are not whole there)
  if (a.M > 1 && !within_reach(a.M, a.lda, a.K)) {
    GemmArgs low = a, high = a;
    const int64_t m = low.M = a.M / 2;
    high.M = a.M - low.M;
    high.A = static_cast<const uint16_t*>(a.A) + m * a.lda;
    if (a.residual) high.residual = a.residual + m * a.ldc;
    if (a.C) high.C = a.C + m * a.ldc;
    if (a.C2) high.C2 = static_cast<char*>(a.C2) + m * a.ldc2 * (a.c2_dtype == DH_F32 ? 4 : 2);
    const int rc = dense_16bit(op, low, f16);
    return rc ? rc : dense_16bit(op, high, f16);
  }
  if (a.N > 1 && !within_reach(a.N, a.ldw, a.K)) {
    GemmArgs low = a, high = a;
    const int n = low.N = a.N / 2;
    high.N = a.N - n;
    low.n_first = std::min(a.n_first, n);
    high.n_first = a.n_first - low.n_first;
    high.W = a.W + (int64_t)n * a.ldw;
    if (a.bias) high.bias = a.bias + n;
    if (a.col_scale) high.col_scale = a.col_scale + n;
    if (a.residual) high.residual = a.residual + n;
    if (a.C) high.C = a.C + n;
    if (a.C2) high.C2 = static_cast<char*>(a.C2) + (int64_t)(n - low.n_first) * (a.c2_dtype == DH_F32 ? 4 : 2);
    const int rc = dense_16bit(op, low, f16);
    return rc ? rc : dense_16bit(op, high, f16);
  }
  return launch_act(op, a, f16, choose_16bit(a.M, a.N, a.K, a.n_first < a.N && a.act == DH_ACT_GELU_ERF));
}

// Tiles of the 32-bit products, and their costs as above, fitted to 318 products (M 2 .. 2048, N 64 .. 20000, K 64 .. 16384) with each tile and
// up to 16 slices, weights from HBM: the choice is 0.7 % behind the best on average, 15 % at worst.
using Split32x64 = dh::SplitTile<1, 2, 4, 4, 2>;
using Split64x64 = dh::SplitTile<2, 2, 4, 3, 4>;
using Split128x128 = dh::SplitTile<4, 4, 2, 3, 2>;
constexpr TileCost kSplitTiles[] = {{32, 64, 2, 201.f, 287.f, 503.f, 4500.f, 2730.f},
                                    {64, 64, 2, 304.f, 411.f, 800.f, 4730.f, 2600.f},
                                    {128, 128, 1, 737.f, 1190.f, 1293.f, 9470.f, 7970.f}};
constexpr int kSplitK = 128;                     // two steps
TileChoice choose_f32(int64_t M, int64_t N, int64_t K) {
  const int64_t steps = K / 64;
  const int most = slices_in_workspace(M, N, kMaxSlices);
  TileChoice best{0, 1};
  double least = 1e30;
  for (int i = 0; i < 3; i++)
    for (int s = 1; s <= most && (s == 1 || steps / s >= 2); s++) {
      const TileCost& c = kSplitTiles[i];
      const int64_t groups = dh::ceil_div(M, c.bm) * dh::ceil_div(N, c.bn) * s;
      double t = std::max(loops_ns(c, groups, dh::ceil_div(steps, s), 0.9), 2.0 * N * K / 6165.0) + c.start;
      if (s > 1) t += 2450.0 + 4.0 * M * N * (2 * s + 1) / 6300.0;
      if (t < least) {
        least = t;
        best = TileChoice{i, s};
      }
    }
  const int env_tile = dh::tuning_int("DH_F32_TILE", -1), env_slices = dh::tuning_int("DH_F32_SLICES", 0);
  if (env_tile >= 0) best.tile = env_tile;
  if (env_slices) best.slices = std::min(most, env_slices);
  return best;
}
// k slices of a product that goes through registers.  Workgroups on a compute unit share its matrix cores, so the one with the most of them
// ends last: 64 k of a tile take 1.35 us alone there and 1.1 us each in company (0.85 at the full rate).  Slices cost a launch and 4 bytes a sum
// at 4 TB/s.
int choose_register_slices(int64_t M, int64_t N, int64_t K) {
  const int64_t steps = K / 64, tiles = dh::ceil_div(M, 64) * dh::ceil_div(N, 64);
  const int most = slices_in_workspace(M, N, kMaxSlices);
  int slices = 1;
  double least = 1e30;
  for (int s = 1; s <= most && (s == 1 || steps / s >= 2); s++) {
    const int64_t together = dh::ceil_div(tiles * s, dh::num_cus());
    double t = (together == 1 ? 1350.0 : 1100.0 * together) * dh::ceil_div(steps, s);
    if (s > 1) t += 3500.0 + 4.0 * M * N * (2 * s + 1) / 4000.0;
    if (t < least) {
      least = t;
      slices = s;
    }
  }
  return slices;
}

template <class Tile>
int launch_split(const char* op, GemmArgs a, int slices) {
  auto kern = gemm_split_kernel<Tile>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::kLds);
  DH_CHECK_HIP(op, set);
  a.tiles_m = (int)dh::ceil_div(a.M, Tile::BM);
  a.tiles_n = (int)dh::ceil_div(a.N, Tile::BN);
  hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)a.tiles_m * a.tiles_n), slices), dim3(Tile::kThreads), Tile::kLds, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}
// Rows below 4 GB apart within a tile and at least two steps take the bf16 matrix cores.  A single step has nothing to hide its start
// behind: 361 x 8204 x 64 takes 9.4 us with 32-bit instructions and 12.1 without, 2024 x 3594 x 64 17.9 and 21.9; at two steps bf16
// takes 0.96 of the other's time on average (1.13 at worst, 63 x 12699 x 128), at three 0.81, at four 0.70.
int dense_f32(const char* op, GemmArgs a) {
  const bool split = a.K >= kSplitK && 4 * (std::min<int64_t>(a.M, Split128x128::BM) * a.lda + a.K) < (int64_t)1 << 32 && within_reach(a.N, a.ldw, a.K);
  const TileChoice pick = split ? choose_f32(a.M, a.N, a.K) : TileChoice{0, choose_register_slices(a.M, a.N, a.K)};
  a.k_slice = slice_extent(a.K, pick.slices);
  const int slices = (int)dh::ceil_div(a.K, a.k_slice);
  size_t ws_bytes = 0;
  if (slices > 1) a.parts = dh::splitk_workspace(&ws_bytes);
  if (!split) {
    a.tiles_m = (int)dh::ceil_div(a.M, 64);
    a.tiles_n = (int)dh::ceil_div(a.N, 64);
    hipLaunchKernelGGL((gemm_f32_kernel<1, false, false>), dim3((unsigned)((int64_t)a.tiles_m * a.tiles_n), slices), dim3(256), 0, dh::stream(), a);
    DH_CHECK_LAUNCH(op);
  } else {
    const int rc = pick.tile == 0 ? launch_split<Split32x64>(op, a, slices)
                 : pick.tile == 1 ? launch_split<Split64x64>(op, a, slices)
                                  : launch_split<Split128x128>(op, a, slices);
    if (rc) return rc;
  }
  return slices > 1 ? launch_reduce(op, a, slices) : 0;
}

// Expert products; the grouped ones launch as many row tiles as the table has room for.
template <bool GROUPED, bool GLU>
int launch_experts(const char* op, GemmArgs a, int a_dtype) {
  a.k_slice = a.K;
  if (a_dtype == DH_F32) {
    constexpr int TN = GLU ? 2 : 1;
    a.tiles_n = (int)dh::ceil_div(a.N, 64 * TN);
    if (!GROUPED) a.tiles_m = (int)dh::ceil_div(a.M, 64);
    hipLaunchKernelGGL((gemm_f32_kernel<TN, GROUPED, GLU>), dim3(a.tiles_m * a.tiles_n), dim3(256), 0, dh::stream(), a);
    DH_CHECK_LAUNCH(op);
    return 0;
  }
  if constexpr (GROUPED) {
    if (a.rows.tile_rows == Tile128x128::BM) return launch_16bit_kernel<Tile128x128, false, kNoSecond, true, GLU>(op, a, 1);
    return launch_16bit_kernel<std::conditional_t<GLU, Tile64x128, Tile64x64>, false, kNoSecond, true, GLU>(op, a, 1);
  } else {
    return launch_16bit<false, kNoSecond, GLU>(op, a, choose_tile(a.M, a.N, a.K, 1, true, false));
  }
}

template <class Tile, bool GLU>
int launch_pair(const char* op, GemmArgs shared, GemmArgs routed) {
  auto kern = gemm_experts_kernel<Tile, GLU>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::kLds);
  DH_CHECK_HIP(op, set);
  shared.tiles_m = (int)dh::ceil_div(shared.M, Tile::BM);
  shared.tiles_n = (int)dh::ceil_div(shared.N, Tile::BN);
  routed.tiles_n = (int)dh::ceil_div(routed.N, Tile::BN);
  const int own = (int)dh::ceil_div((int64_t)shared.tiles_m * shared.tiles_n, 8) * 8;
  hipLaunchKernelGGL(kern, dim3(own + routed.tiles_m * routed.tiles_n), dim3(Tile::kThreads), Tile::kLds, dh::stream(), shared, routed, own);
  DH_CHECK_LAUNCH(op);
  return 0;
}
GemmArgs expert_args(const dh::ExpertProduct& p, bool glu) {
  GemmArgs a{};
  a.A = p.A; a.W = p.W; a.lda = p.lda; a.ldw = p.ldw; a.M = p.M; a.N = p.N; a.K = a.k_slice = p.K; a.alpha = 1.f; a.rows = p.rows;
  a.tiles_m = p.rows.max_tiles;
  if (glu) {
    a.C2 = p.out; a.c2_dtype = DH_BF16; a.ldc2 = (int)p.ld_out;
  } else {
    a.C = static_cast<float*>(p.out); a.ldc = (int)p.ld_out; a.n_first = p.N;
  }
  return a;
}

}  // namespace

namespace dh {

// One launch where neither product is small beside the other and the shared one loses little on the routed ones' tiles (what the shared last round
// gains is not weighed against that loss).  Each fills one to two rounds of workgroups and leaves most of its last round empty, together they leave one:
// apart and together, us, the gate and up products and the down products of prompts of 2000 rows of 1024: 25.7 + 22.1 to 45.1, 24.9 + 17.0 to 31.1; 1531 of
// 2048: 65.6 + 52.2 to 102, 48.2 + 31.5 to 66 (and 1 more in the launch that sums); 900 of 4096: 130 + 105 to 220, 92 + 50 to 143.  Whole layers of experts, widths
// 1024 to 4096, 2 to 2047 rows, by this rule against all apart on tiles that did not ask for their weights ahead: 0.99 to 1.41 times as fast.
bool experts_together(const ExpertProduct& routed, const ExpertProduct& shared, bool glu) {
  const int at = routed.rows.tile_rows == Tile128x128::BM ? 2 : 3;
  const TileCost& c = glu ? kGluTiles[at] : kTiles[at];
  const double work[2] = {(double)routed.M * routed.N * routed.K, (double)shared.M * shared.N * shared.K};
  if (4.0 * std::min(work[0], work[1]) < std::max(work[0], work[1])) return false;
  // (gate and up products gather their rows)
  if (!(glu ? (int64_t)2 * routed.rows.source_rows * routed.lda < (int64_t)1 << 32 : within_reach(c.bm, routed.lda, routed.K)) ||
      !within_reach(routed.N, routed.ldw, routed.K) || !within_reach(shared.M, shared.lda, shared.K) || !within_reach(shared.N, shared.ldw, shared.K))
    return false;
  const int64_t tiles_n = dh::ceil_div(routed.N, c.bn), own = dh::ceil_div(shared.M, c.bm) * dh::ceil_div(shared.N, c.bn);
  if ((own + 8 + routed.rows.max_tiles * tiles_n) * 256 >= (int64_t)1 << 32) return false;   // threads of one launch
  if (!glu && (dh::tuning_int("DH_DENSE_TILE", -1) >= 0 || dh::tuning_int("DH_DENSE_SLICES", 0))) return false;     // asked for by name: apart, as asked
  const TileChoice best = glu ? choose_tile(shared.M, shared.N, shared.K, 1, true, false) : choose_16bit(shared.M, shared.N, shared.K, false);
  // (slices of the shared one would be sums in another order)
  return best.slices == 1 && loops_ns(c, own, shared.K / 64, 0.76) + c.start <= 1.15 * best.ns;
}
int experts_pair(const char* op, const ExpertProduct& routed, const ExpertProduct& shared, bool glu) {
  const GemmArgs r = expert_args(routed, glu), s = expert_args(shared, glu);
  if (routed.rows.tile_rows == Tile128x128::BM) return glu ? launch_pair<Tile128x128, true>(op, s, r) : launch_pair<Tile128x128, false>(op, s, r);
  return glu ? launch_pair<Tile64x128, true>(op, s, r) : launch_pair<Tile64x64, false>(op, s, r);
}

int expert_tile_rows(int a_dtype, int rows, int groups) { return a_dtype == DH_F32 || rows < 96 * groups ? 64 : Tile128x128::BM; }

int experts_glu(const char* op, const ExpertRows& rows, const void* A, int a_dtype, int64_t lda, const uint16_t* W, int64_t ldw, int M,
                int N, int K, void* out, int out_dtype, int64_t ld_out) {
  GemmArgs a{};
  a.A = A; a.W = W; a.lda = lda; a.ldw = ldw; a.M = M; a.N = N; a.K = K; a.alpha = 1.f;
  a.C2 = out; a.c2_dtype = out_dtype; a.ldc2 = (int)ld_out; a.rows = rows;
  if (rows.tiles) {
    a.tiles_m = rows.max_tiles;
    return launch_experts<true, true>(op, a, a_dtype);
  }
  return launch_experts<false, true>(op, a, a_dtype);
}

int experts_down(const char* op, const ExpertRows& rows, const void* A, int a_dtype, int64_t lda, const uint16_t* W, int64_t ldw, int N,
                 int K, float* out, int64_t ld_out) {
  GemmArgs a{};
  a.A = A; a.W = W; a.lda = lda; a.ldw = ldw; a.N = N; a.K = K; a.alpha = 1.f;
  a.C = out; a.ldc = (int)ld_out; a.n_first = N; a.rows = rows;
  a.tiles_m = rows.max_tiles;
  return launch_experts<true, false>(op, a, a_dtype);
}

}  // namespace dh

extern "C" int dh_dense_matmul(const void* d_A, int a_dtype, int lda, const void* d_W, int ldw, int M, int N, int K,
                               float alpha, const float* d_bias, const float* d_residual, float* d_C, int ldc, int n_first,
                               void* d_C2, int c2_dtype, int ldc2, int activation) {
  return dh_dense_matmul_scaled(d_A, a_dtype, lda, d_W, ldw, M, N, K, alpha, d_bias, nullptr, d_residual, d_C, ldc, n_first, d_C2,
                                c2_dtype, ldc2, activation);
}

static int dense_matmul(const char* op, const void* d_A, int a_dtype, int lda, const void* d_W, int ldw, int M, int N, int K,
                        float alpha, const float* d_bias, const float* d_col_scale, const float* d_residual,
                        float* d_C, int ldc, int n_first, void* d_C2, int c2_dtype, int ldc2, int activation, const GemmArgs& norm) {
  DH_REQUIRE_INIT(op);
  if (M <= 0 || N <= 0 || K <= 0) return dh::fail(1, "[%s] Dimensions must be positive: M=%d, N=%d, K=%d", op, M, N, K);
  if (K % 64) return dh::fail(1, "[%s] K=%d must be a multiple of 64 (zero-padded)", op, K);
  if (lda < K || ldw < K || lda % 8 || ldw % 8)
    return dh::fail(1, "[%s] row strides must be multiples of 8 and hold K=%d elements (lda=%d, ldw=%d)", op, K, lda, ldw);
  if (a_dtype != DH_BF16 && a_dtype != DH_F32 && a_dtype != DH_F16)
    return dh::fail(1, "[%s] activations must be bf16, f16 (with f16 weights) or f32, got dtype %d", op, a_dtype);
  if (n_first < 0 || n_first > N) return dh::fail(1, "[%s] n_first=%d is outside 0..%d", op, n_first, N);
  if (!d_A || !d_W || (n_first > 0 && !d_C) || (n_first < N && !d_C2)) return dh::fail(1, "[%s] null pointer", op);
  if (n_first > 0 && ldc < n_first) return dh::fail(1, "[%s] ldc=%d is shorter than %d columns", op, ldc, n_first);
  if (n_first < N && (ldc2 < N - n_first || (c2_dtype != DH_BF16 && c2_dtype != DH_F16 && c2_dtype != DH_F32)))
    return dh::fail(1, "[%s] the second output needs %d columns of bf16, f16 or f32 (ldc2=%d, dtype %d)", op, N - n_first, ldc2, c2_dtype);
  if ((reinterpret_cast<uintptr_t>(d_A) | reinterpret_cast<uintptr_t>(d_W)) & 15)
    return dh::fail(1, "[%s] activation and weight pointers must be 16-byte aligned", op);
  GemmArgs a = norm;
  a.A = d_A; a.W = static_cast<const uint16_t*>(d_W); a.lda = lda; a.ldw = ldw;
  a.M = M; a.N = N; a.K = K; a.alpha = alpha; a.bias = d_bias; a.residual = d_residual; a.col_scale = d_col_scale;
  a.C = d_C; a.ldc = ldc; a.n_first = n_first;
  a.C2 = d_C2; a.ldc2 = ldc2; a.c2_dtype = c2_dtype; a.act = activation;
  if (a_dtype == DH_F32) return dense_f32(op, a);
  return dense_16bit(op, a, a_dtype == DH_F16);
}

extern "C" int dh_dense_matmul_scaled(const void* d_A, int a_dtype, int lda, const void* d_W, int ldw, int M, int N, int K,
                                      float alpha, const float* d_bias, const float* d_col_scale, const float* d_residual,
                                      float* d_C, int ldc, int n_first, void* d_C2, int c2_dtype, int ldc2, int activation) {
  return dense_matmul("dh_dense_matmul", d_A, a_dtype, lda, d_W, ldw, M, N, K, alpha, d_bias, d_col_scale, d_residual, d_C, ldc, n_first, d_C2, c2_dtype, ldc2,
                      activation, GemmArgs{});
}

extern "C" int dh_dense_matmul_normed(const void* d_A, int a_dtype, int lda, const void* d_W, int ldw, int M, int N, int K, const float* d_col_scale,
                                      const float* d_residual, float* d_C, int ldc, const float* d_norm_weight, float eps, void* d_normed, int normed_dtype,
                                      int ld_normed) {
  const char* op = "dh_dense_matmul_normed";
  DH_REQUIRE_INIT(op);
  if (normed_dtype != DH_BF16 && normed_dtype != DH_F32) return dh::fail(1, "[%s] normed rows must be bf16 or f32, got dtype %d", op, normed_dtype);
  if (!d_norm_weight || !d_normed) return dh::fail(1, "[%s] null pointer", op);
  if (ld_normed < N || !(eps >= 0.f)) return dh::fail(1, "[%s] normed rows of %d do not hold %d elements, or eps is negative", op, ld_normed, N);
  if ((reinterpret_cast<uintptr_t>(d_norm_weight) | reinterpret_cast<uintptr_t>(d_normed) | reinterpret_cast<uintptr_t>(d_C)) & 15)
    return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  bool done = false;
  GemmArgs norm{};
  norm.norm_weight = d_norm_weight; norm.norm_eps = eps; norm.normed = d_normed; norm.normed_dtype = normed_dtype; norm.ld_normed = ld_normed; norm.norm_done = &done;
  if (int rc = dense_matmul(op, d_A, a_dtype, lda, d_W, ldw, M, N, K, 1.f, nullptr, d_col_scale, d_residual, d_C, ldc, N, nullptr, 0, 0, DH_ACT_NONE, norm)) return rc;
  return done ? 0 : dh_rmsnorm_rows(d_C, ldc, nullptr, d_norm_weight, d_normed, normed_dtype, ld_normed, M, N, eps);
}

extern "C" int dh_dense_matmul_layout(int M, int N, int K, int a_dtype, int form, int num_cus, int64_t* out3) {
  const char* op = "dh_dense_matmul_layout";
  if (!out3 || M <= 0 || N <= 0 || K <= 0 || K % 64) return dh::fail(1, "[%s] M=%d, N=%d, K=%d (a multiple of 64), or no place for the result", op, M, N, K);
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  const bool wide = a_dtype == DH_F32, glu = form == 1;
  const bool registers = wide && (glu || K < kSplitK || form == 3);
  const TileChoice pick = registers ? TileChoice{0, glu ? 1 : choose_register_slices(M, N, K)} : wide ? choose_f32(M, N, K) : glu ? choose_tile(M, N, K, 1, true, false) : choose_16bit(M, N, K, form == 2);
  dh::plan_end();
  const TileCost& c = wide ? kSplitTiles[pick.tile] : glu ? kGluTiles[pick.tile] : kTiles[pick.tile];
  out3[0] = registers ? 64 : c.bm;
  out3[1] = registers ? (glu ? 128 : 64) : c.bn;
  out3[2] = dh::ceil_div(K, slice_extent(K, pick.slices));
  return 0;
}
