// Matrix memory with exponential gates (dh_mlstm): per head a state S [dim][vdim], a normaliser n [dim] and a running maximum m,
//
//   m' = max(f + m, i);  S' = e^(f + m - m') S + e^(i - m') k v^T;  n' likewise with k alone
//   o  = S'^T q / (max(|n' . q|, e^-m') + 1e-6)
//   i  = cap tanh(z_i / cap),  f = log sigmoid(cap tanh(z_f / cap)),  m starts at 0
//
// everything in 32-bit.  S is updated in place; n and m live in two slots, and a step at position p reads slot p & 1 and
// writes the other, so that every workgroup of a head can read them while one writes.  At position 0 the state counts as zero,
// whatever the buffers hold.
//
// Decode: mlstm_step_kernel, one workgroup per (head, 32 value columns).
// Prefill cuts a portion into chunks of 64 tokens.  With F the running sum of f (kept in double: its differences are the
// exponents), m is known for every token from a max-plus scan, and a chunk's outputs are a product with the state before it plus a
// masked product inside it:
//
//   mlstm_gates_kernel     F, i, m of every token, one workgroup per head; beside them every chunk's scores Q K^T
//   mlstm_states_kernel    the state in front of every chunk, walking the chunks with a tile of it in registers; or, where few tiles would
//                          walk far, in two launches:
//   mlstm_chunks_kernel    what every chunk adds to the state behind it, sum_s e^(F_end - F_s + i_s - m_end) k_s v_s^T: independent of
//                          one another, because m is known
//   mlstm_scan_kernel      the state in front of every chunk, S_(c+1) = e^(F_end - F_start + m_start - m_end) S_c + what chunk c adds,
//                          element by element and in place
//   mlstm_outputs_kernel   o of (chunk, head, value columns): Q S, decay and mask of the scores, then (Q K^T) V
//
// on the 32-bit matrix-core instructions v_mfma_f32_32x32x2_f32 and, in the walk, v_mfma_f32_16x16x4_f32 (which add in the same order).
// head_norm_gate_kernel then divides every head's output by its root mean square and applies the weight and the output gate.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "gemm_wide.h"

namespace {

using dh::f32x16_t;
using dh::f32x4_t;

constexpr int kChunk = 64;           // tokens per chunk
constexpr int kCols = 32;            // value columns per workgroup of a step
constexpr float kDenominatorEps = 1e-6f;

struct MemArgs {
  const float* rows;       // projection rows [T][ld_row]: q heads, k heads, v heads, .., i, f
  float* S;                // [H][DP][VP]
  float* n;                // [2][H][DP]
  float* m;                // [2][H]
  float* out;              // [T][ld_out] raw head outputs
  int64_t ld_row, ld_out;
  int H, DP, VP, k_off, v_off, i_off, f_off;
  float gate_cap, q_scale;
  int pos, T, chunks;
  const uint32_t* kv_len;
  // portions: gates [H][T], states in front of chunks
  double* F;
  float* i;
  float* mt;               // m after every token
  float* mc;               // [H][chunks + 1] m in front of every chunk, and at the end
  float* keep;             // [H][chunks] what a chunk leaves of the state in front of it
  float* w;                // [H][chunks][64] weight of a token's key and value in the state behind its chunk, zero past the last; null: no walk
  float* scores;           // [chunks][H][64][64] q . k of a chunk's tokens, not decayed; nothing past the diagonal's 16 x 16 tiles
  float* Sc;               // [chunks + 1][H][DP][VP]
  float* nc;               // [chunks + 1][H][DP]
};

__device__ __forceinline__ float log_input_gate(const MemArgs& a, float z) { return a.gate_cap * tanhf(z / a.gate_cap); }
__device__ __forceinline__ float log_forget_gate(const MemArgs& a, float z) {
  const float t = a.gate_cap * tanhf(z / a.gate_cap);
  return fminf(t, 0.f) - log1pf(expf(-fabsf(t)));
}

// Eight lanes x four columns, 32 rows at a time.  Four heads of 128 x 256: 5.3 -> 4.0 us with what 128 rows need requested in front of the gates.
__global__ __launch_bounds__(256) void mlstm_step_kernel(const MemArgs a) {
  __shared__ float red[4];
  __shared__ float4 o_lds[4][8];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y, col = kCols * blockIdx.x + 4 * (tid & 7);
  const int pos = a.kv_len ? max(0, (int)*a.kv_len - 1) : a.pos;
  const bool first = pos == 0;
  const int from = pos & 1, to = from ^ 1;
  const float* q = a.rows + (int64_t)h * a.DP;
  const float* k = a.rows + a.k_off + (int64_t)h * a.DP;
  // what the first four rows of a thread need is requested before anything is computed from it: one trip to memory up to 128 rows (a longer state's
  // next four are requested behind the stores of these)
  constexpr int BATCH = 4;
  float* S = a.S + (int64_t)h * a.DP * a.VP + col;
  const float* n_old = a.n + ((int64_t)from * a.H + h) * a.DP;
  float* n_new = a.n + ((int64_t)to * a.H + h) * a.DP;
  float4 s[BATCH];
  float kr[BATCH], qr[BATCH];
  auto request = [&](int r0) {
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int r = min(r0 + 32 * b, a.DP - 1);
      s[b] = *reinterpret_cast<const float4*>(S + (int64_t)r * a.VP);
      kr[b] = k[r];
      qr[b] = q[r];
    }
  };
  const float zi = a.rows[a.i_off + h], zf = a.rows[a.f_off + h], m_held = a.m[from * a.H + h];
  const float4 v = *reinterpret_cast<const float4*>(a.rows + a.v_off + (int64_t)h * a.VP + col);
  request(tid >> 3);
  const int nr = min(tid, a.DP - 1);
  float n_r = n_old[nr], nk = k[nr], nq = q[nr];
  const float li = log_input_gate(a, zi), lf = log_forget_gate(a, zf);
  const float m_old = first ? 0.f : m_held;
  const float m_new = fmaxf(lf + m_old, li);
  const float keep = first ? 0.f : expf(lf + m_old - m_new), put = expf(li - m_new);

  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int r0 = tid >> 3; r0 < a.DP; r0 += 32 * BATCH) {
    if (r0 != tid >> 3) request(r0);
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int r = r0 + 32 * b;
      if (r >= a.DP) break;
      float4 y = first ? make_float4(0.f, 0.f, 0.f, 0.f) : s[b];
      const float kp = put * kr[b];
      y.x = fmaf(keep, y.x, kp * v.x); y.y = fmaf(keep, y.y, kp * v.y);
      y.z = fmaf(keep, y.z, kp * v.z); y.w = fmaf(keep, y.w, kp * v.w);
      *reinterpret_cast<float4*>(S + (int64_t)r * a.VP) = y;
      acc.x = fmaf(qr[b], y.x, acc.x); acc.y = fmaf(qr[b], y.y, acc.y);
      acc.z = fmaf(qr[b], y.z, acc.z); acc.w = fmaf(qr[b], y.w, acc.w);
    }
  }
  float dot = 0.f;
  for (int r = tid; r < a.DP; r += 256) {
    if (r != tid) { n_r = n_old[r]; nk = k[r]; nq = q[r]; }
    const float n = fmaf(keep, first ? 0.f : n_r, put * nk);
    dot = fmaf(n, nq, dot);
    if (blockIdx.x == 0) n_new[r] = n;
  }
  if (blockIdx.x == 0 && tid == 0) a.m[to * a.H + h] = m_new;
  // lanes that hold the same columns lie 8 apart
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) {
    acc.x += __shfl_xor(acc.x, off, 64); acc.y += __shfl_xor(acc.y, off, 64);
    acc.z += __shfl_xor(acc.z, off, 64); acc.w += __shfl_xor(acc.w, off, 64);
  }
  dot = dh::wave_sum_uniform(dot);
  if (lane < 8) o_lds[wave][lane] = acc;
  if (lane == 0) red[wave] = dot;
  __syncthreads();
  if (tid < 8) {
    const float nq = (red[0] + red[1] + red[2] + red[3]) * a.q_scale;
    const float f = a.q_scale / (fmaxf(fabsf(nq), expf(-m_new)) + kDenominatorEps);
    float4 o = o_lds[0][tid];
#pragma unroll
    for (int w = 1; w < 4; w++) { o.x += o_lds[w][tid].x; o.y += o_lds[w][tid].y; o.z += o_lds[w][tid].z; o.w += o_lds[w][tid].w; }
    *reinterpret_cast<float4*>(a.out + (int64_t)h * a.VP + col) = make_float4(o.x * f, o.y * f, o.z * f, o.w * f);
  }
}

// (F, M): a stretch of tokens takes m to max(m + F, M).
struct MaxPlus {
  double F, M;
};
__device__ __forceinline__ MaxPlus then(const MaxPlus& x, const MaxPlus& y) { return {x.F + y.F, fmax(x.M + y.F, y.M)}; }
// Lane l's value becomes that of lanes 0 .. l one after the other (of LANES in a row).
template <int LANES>
__device__ __forceinline__ MaxPlus scan_lanes(MaxPlus v, int lane) {
#pragma unroll
  for (int off = 1; off < LANES; off <<= 1) {
    const MaxPlus up = {__shfl_up(v.F, off, 64), __shfl_up(v.M, off, 64)};
    if (lane >= off) v = then(up, v);
  }
  return v;
}

// One head's gates.  A thread takes a stretch of tokens, four of them at a time; up to four stay in its registers.
constexpr int kHeldChunks = 1024;                      // chunks whose ends stay in LDS
struct GatesLds {
  MaxPlus stretches[16];
  double F_end[kHeldChunks];                           // F of a chunk's last token
  float m_front[kHeldChunks + 1];                      // m in front of it
};
__device__ __forceinline__ void head_gates(const MemArgs& a, int h, GatesLds& lds) {
  constexpr int U = 4;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int per = (a.T + 1023) / 1024, t0 = min(tid * per, a.T), t1 = min(t0 + per, a.T);
  const float m_in = a.pos == 0 ? 0.f : a.m[(a.pos & 1) * a.H + h];
  double* F = a.F + (int64_t)h * a.T;
  float* li = a.i + (int64_t)h * a.T;
  float* mt = a.mt + (int64_t)h * a.T;
  float* mc = a.mc + (int64_t)h * (a.chunks + 1);
  double f[U];                                         // of the four at hand: f, then F
  float i[U];
  MaxPlus run = {0.0, -1e30};
  for (int t = t0; t < t1; t += U) {
    float zf[U], zi[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (u >= per) break;                             // (a line of memory each)
      const float* row = a.rows + (int64_t)min(t + u, a.T - 1) * a.ld_row;
      zf[u] = row[a.f_off + h];
      zi[u] = row[a.i_off + h];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (t + u >= t1) break;
      f[u] = (double)log_forget_gate(a, zf[u]);
      i[u] = log_input_gate(a, zi[u]);
      run = then(run, {f[u], (double)i[u]});
      if (per > U) F[t + u] = f[u];                    // becomes the running sum below
      li[t + u] = i[u];
    }
  }
  // what lies in front of a thread's stretch: the waves before its own, and their lanes before its own
  const MaxPlus upto = scan_lanes<64>(run, lane);
  if (lane == 63) lds.stretches[wave] = upto;
  __syncthreads();
  const MaxPlus waves = scan_lanes<16>(lds.stretches[lane & 15], lane & 15);
  MaxPlus before = {__shfl(waves.F, max(wave - 1, 0), 64), __shfl(waves.M, max(wave - 1, 0), 64)};
  if (wave == 0) before = MaxPlus{0.0, -1e30};
  const MaxPlus own = {__shfl_up(upto.F, 1, 64), __shfl_up(upto.M, 1, 64)};
  if (lane > 0) before = then(before, own);
  double sum = before.F, m = fmax((double)m_in + before.F, before.M);
  auto front = [&](int c) {
    mc[c] = (float)m;
    if (c <= kHeldChunks) lds.m_front[c] = (float)m;
  };
  auto again = [&](int t) {                            // a longer stretch's next four
    if (per > U)
#pragma unroll
      for (int u = 0; u < U; u++) {
        f[u] = F[min(t + u, a.T - 1)];
        i[u] = li[min(t + u, a.T - 1)];
      }
  };
  for (int t = t0; t < t1; t += U) {
    again(t);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (t + u >= t1) break;
      if ((t + u) % kChunk == 0) front((t + u) / kChunk);
      sum += f[u];
      m = fmax(m + f[u], (double)i[u]);
      f[u] = sum;
      F[t + u] = sum;
      mt[t + u] = (float)m;
      const bool last = t + u == a.T - 1;
      if ((last || (t + u) % kChunk == kChunk - 1) && (t + u) / kChunk < kHeldChunks) lds.F_end[(t + u) / kChunk] = sum;
      if (last) {
        front(a.chunks);
        a.m[((a.pos + a.T) & 1) * a.H + h] = (float)m;
      }
    }
  }
  __syncthreads();
  auto F_end = [&](int c) { return c < kHeldChunks ? lds.F_end[c] : F[min((c + 1) * kChunk, a.T) - 1]; };
  auto m_front = [&](int c) { return (double)(c <= kHeldChunks ? lds.m_front[c] : mc[c]); };
  for (int c = tid; c < a.chunks; c += 1024)
    a.keep[(int64_t)h * a.chunks + c] = expf((float)(F_end(c) - (c > 0 ? F_end(c - 1) : 0.0) + m_front(c) - m_front(c + 1)));
  if (!a.w) return;
  // in fours of tokens, a token of every four beside those of the others
  auto put_weight = [&](int t, float w) { a.w[((int64_t)h * a.chunks + t / kChunk) * kChunk + 16 * (t & 3) + ((t & (kChunk - 1)) >> 2)] = w; };
  for (int t = t0; t < t1; t += U) {
    again(t);
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (t + u >= t1) break;
      const int c = (t + u) / kChunk;
      put_weight(t + u, expf((float)(F_end(c) - f[u] + (double)i[u] - m_front(c + 1))));
    }
  }
  for (int t = a.T + tid; t < a.chunks * kChunk; t += 1024) put_weight(t, 0.f);
}

// The scores Q K^T of one (chunk, head), the 16 x 16 tiles up to the diagonal; a wave has one tile of them.
constexpr int kScoreRow = 64 + 4;                      // floats of a row in LDS: sixteen rows' 16-byte pieces lie in different banks
__device__ __forceinline__ void chunk_scores(const MemArgs& a, int item, float* lds) {
  float *qs = lds, *ks = lds + kChunk * kScoreRow;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = item / a.H, h = item % a.H;
  const int first = c * kChunk, x = 4 * (tid & 15), at = (tid >> 4) * kScoreRow + x;
  const float* row = a.rows + (int64_t)(first + min(tid >> 4, a.T - first - 1)) * a.ld_row + (int64_t)h * a.DP;
  constexpr int AHEAD = 4;                             // 64 dims each, requested together
  f32x4_t q[AHEAD], k[AHEAD];
  const int tr = wave < 1 ? 0 : wave < 3 ? 1 : wave < 6 ? 2 : 3, tc = wave - tr * (tr + 1) / 2;
  f32x4_t p = {0.f, 0.f, 0.f, 0.f};
  for (int d = 0; d < a.DP; d += 64 * AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      const int du = min(d + 64 * u + x, a.DP - 4);
      q[u] = *reinterpret_cast<const f32x4_t*>(row + du);
      k[u] = *reinterpret_cast<const f32x4_t*>(row + a.k_off + du);
    }
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      const int d0 = d + 64 * u;
      if (d0 >= a.DP) break;
      if (d0 + x >= a.DP) q[u] = k[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
      *reinterpret_cast<f32x4_t*>(qs + at) = q[u] * a.q_scale;
      *reinterpret_cast<f32x4_t*>(ks + at) = k[u];
      __syncthreads();
      if (wave < 10) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int place = 16 * s + 4 * (lane >> 4);
          const f32x4_t fq = *reinterpret_cast<const f32x4_t*>(qs + (16 * tr + (lane & 15)) * kScoreRow + place);
          const f32x4_t fk = *reinterpret_cast<const f32x4_t*>(ks + (16 * tc + (lane & 15)) * kScoreRow + place);
#pragma unroll
          for (int e = 0; e < 4; e++) p = __builtin_amdgcn_mfma_f32_16x16x4f32(fq[e], fk[e], p, 0, 0, 0);
        }
      }
    }
  }
  if (wave < 10) {
    float* to = a.scores + (int64_t)item * (kChunk * kChunk) + (16 * tr + 4 * (lane >> 4)) * kChunk + 16 * tc + (lane & 15);
#pragma unroll
    for (int e = 0; e < 4; e++) to[e * kChunk] = p[e];
  }
}

// Grid = (chunks + 1, heads).  The first H workgroups: the heads' gates, a chain of short steps; the others, meanwhile: a chunk's and head's scores, which need no gate.
// us, four heads of 256 x 512, 1531 tokens: gates alone 11.3 (three trips to memory for a second token, which are one
// now), both 9.4, the scores by themselves 6.4 of that.
__global__ __launch_bounds__(1024) void mlstm_gates_kernel(const MemArgs a) {
  __shared__ __align__(16) float lds[2 * kChunk * kScoreRow];
  static_assert(sizeof(GatesLds) <= sizeof(lds), "either of them");
  const int block = blockIdx.x + gridDim.x * blockIdx.y;
  if (block < a.H) head_gates(a, block, *reinterpret_cast<GatesLds*>(lds));
  else chunk_scores(a, block - a.H, lds);
}

// Grid = (64 x 64 tiles of a head's state, heads, chunks); wave w: rows 32 (w >> 1), columns 32 (w & 1) of the tile.
__global__ __launch_bounds__(256) void mlstm_chunks_kernel(const MemArgs a) {
  constexpr int ROW = 64 + 4;
  __shared__ __align__(16) float ks[kChunk * ROW];     // weighted keys [token][dim]
  __shared__ __align__(16) float vs[kChunk * ROW];     // values [token][column]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y, c = blockIdx.z;
  const int tiles_v = (a.VP + 63) / 64, d0 = 64 * (blockIdx.x / tiles_v), v0 = 64 * (blockIdx.x % tiles_v);
  const double* F = a.F + (int64_t)h * a.T;
  const int first = c * kChunk, count = min(kChunk, a.T - first);
  const double F_end = F[first + count - 1];
  const float m_end = a.mc[(int64_t)h * (a.chunks + 1) + c + 1];
  f32x4_t kr[4], vr[4];
  float w[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int p = tid + 256 * r, tok = first + min(p >> 4, count - 1), x = 4 * (p & 15);
    const float* row = a.rows + (int64_t)tok * a.ld_row;
    kr[r] = vr[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (d0 + x < a.DP) kr[r] = *reinterpret_cast<const f32x4_t*>(row + a.k_off + (int64_t)h * a.DP + d0 + x);
    if (v0 + x < a.VP) vr[r] = *reinterpret_cast<const f32x4_t*>(row + a.v_off + (int64_t)h * a.VP + v0 + x);
    w[r] = (p >> 4) < count ? expf((float)(F_end - F[tok] + (double)a.i[(int64_t)h * a.T + tok] - (double)m_end)) : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int p = tid + 256 * r, tok = p >> 4, x = 4 * (p & 15);
    // (rows past the last repeat it: an infinite one times a weight of zero is no number)
    if ((p >> 4) < count) kr[r] *= w[r];
    else kr[r] = vr[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f32x4_t*>(&ks[tok * ROW + x]) = kr[r];
    *reinterpret_cast<f32x4_t*>(&vs[tok * ROW + x]) = vr[r];
  }
  __syncthreads();
  const int wd = 32 * (wave >> 1), wv = 32 * (wave & 1);
  if (d0 + wd < a.DP && v0 + wv < a.VP) {              // wave-uniform (sizes are multiples of 32)
    f32x16_t acc;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.f;
#pragma unroll 8
    for (int j = 0; j < kChunk / 2; j++) {
      const int tok = 2 * j + (lane >> 5);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ks[tok * ROW + wd + (lane & 31)], vs[tok * ROW + wv + (lane & 31)], acc, 0, 0, 0);
    }
    // accumulator element e of a lane: state row 8 (e / 4) + 4 (lane >> 5) + e % 4, column lane & 31
    float* U = a.Sc + ((int64_t)(c + 1) * a.H + h) * a.DP * a.VP + (int64_t)(d0 + wd + 4 * (lane >> 5)) * a.VP + v0 + wv + (lane & 31);
#pragma unroll
    for (int e = 0; e < 16; e++) U[(int64_t)(8 * (e >> 2) + (e & 3)) * a.VP] = acc[e];
  }
  if (v0 == 0 && tid < 64 && d0 + tid < a.DP) {
    float s = 0.f;
#pragma unroll 8
    for (int t = 0; t < kChunk; t++) s += ks[t * ROW + tid];
    a.nc[((int64_t)(c + 1) * a.H + h) * a.DP + d0 + tid] = s;
  }
}

// Grid = (groups of 1024 elements of a head's [S | n], heads), four per thread; slot 0 of Sc and nc is filled here.
__global__ __launch_bounds__(256) void mlstm_scan_kernel(const MemArgs a) {
  constexpr int AHEAD = 16;
  const int h = blockIdx.y, size = a.DP * a.VP;
  const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= size + a.DP) return;
  const bool is_n = i >= size;
  const int64_t stride = is_n ? (int64_t)a.H * a.DP : (int64_t)a.H * size;
  float* at = is_n ? a.nc + (int64_t)h * a.DP + (i - size) : a.Sc + (int64_t)h * size + i;
  const int64_t slots = (int64_t)a.H * a.DP;
  const float* from = is_n ? a.n + (a.pos & 1) * slots + (int64_t)h * a.DP + (i - size) : a.S + (int64_t)h * size + i;
  float* to = is_n ? a.n + ((a.pos + a.T) & 1) * slots + (int64_t)h * a.DP + (i - size) : a.S + (int64_t)h * size + i;
  const float* keep = a.keep + (int64_t)h * a.chunks;
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (a.pos > 0) s = *reinterpret_cast<const f32x4_t*>(from);
  *reinterpret_cast<f32x4_t*>(at) = s;
  for (int c0 = 0; c0 < a.chunks; c0 += AHEAD) {
    f32x4_t u[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; k++)
      if (c0 + k < a.chunks) u[k] = *reinterpret_cast<const f32x4_t*>(at + (c0 + k + 1) * stride);
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
      const int c = c0 + k;
      if (c < a.chunks) {
        s = s * keep[c] + u[k];
        if (c + 1 < a.chunks) *reinterpret_cast<f32x4_t*>(at + (c + 1) * stride) = s;
      }
    }
  }
  *reinterpret_cast<f32x4_t*>(to) = s;
}

// The states in front of every chunk, S_(c+1) = e^(F_end - F_start + m_start - m_end) S_c + sum_s e^(F_end - F_s + i_s - m_end) k_s v_s^T, in one walk.
//
// One workgroup of eight (four) waves for 64 x 32 (32 x 32) of a head's state, a head's tiles on one die.  Wave w holds rows 16 (w >> 1), columns
// 16 (w & 1) in registers, adds up a chunk's products apart from it (16 of v_mfma_f32_16x16x4_f32: of 32 x 32 for a wave half of the SIMDs would have
// none) and writes the state in front of every chunk once.  Keys, values and weights go straight into three buffers of LDS, two chunks ahead of the one
// being read, by waits that count: through registers the compiler waited for the youngest load and store at every chunk (2.3 us each).  Four tokens make an instruction, so their
// rows' 16-byte pieces are kept apart by 16 banks (slot = piece ^ 4 (token & 3) of 16, piece ^ 4 (token / 2 & 1) of 8).
// The workgroups behind the tiles walk the normaliser.
// us, against a launch for what every chunk adds (to memory and back) and another for the scan: four heads of 256 x 512, 1500 tokens 37.7 + 18.1 -> 33, eight, 1000
// tokens 46 + 21.7 -> 38.5, four of 128 x 256, 2048 tokens 17.2 + 11.4 -> 24.7, 40 tokens 6 + 4.8 -> 4.9.  Of 33 the matrix cores take 15.
template <int ROWS>
struct StateTile {           // ROWS x 32 of a state; a wave 16 x 16 of it
  static constexpr int kWaves = ROWS / 8, kThreads = 64 * kWaves;
  static constexpr int kKeys = kChunk * ROWS * 4, kValues = kChunk * 32 * 4, kBuffer = kKeys + kValues, kBuffers = 3;
  static constexpr int kPieces = ROWS / 4, kKeyTokens = 64 / kPieces, kKeyFetches = kChunk / (kKeyTokens * kWaves);      // of a fetch, of a wave
  static constexpr int kValueFetches = kChunk / (8 * kWaves), kFetches = kKeyFetches + kValueFetches + 1;
  static constexpr int kWeights = kBuffers * kBuffer, kBytes = kWeights + 4 * kChunk * 4;      // four chunks' weights
  // 16-byte piece p of a token's keys (values) lies at slot p ^ key_swap (value_swap)
  static __device__ __forceinline__ int key_swap(int token) { return ROWS == 64 ? 4 * (token & 3) : 4 * ((token >> 1) & 1); }
  static __device__ __forceinline__ int value_swap(int token) { return 4 * ((token >> 1) & 1); }
};
// 64 elements of a head's normaliser: a wave sums a chunk's weighted keys, rounded and added token by token as mlstm_chunks_kernel does, then
// every wave takes the waves' chunks in turn and stores the one in front of which is its own.  The next chunks' keys are requested in front of that.
template <int WAVES>
__device__ __forceinline__ void walk_normaliser(const MemArgs& a, int part, float* sums) {      // [2][WAVES][64]
  constexpr int HALF = kChunk / 2;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int parts = (a.DP + 63) / 64, h = part / parts, d = 64 * (part % parts) + lane;
  const int64_t slots = (int64_t)a.H * a.DP, at = (int64_t)h * a.DP + min(d, a.DP - 1);
  const float* rows = a.rows + a.k_off + (int64_t)h * a.DP + 64 * (part % parts);
  const uint32_t column = (uint32_t)min(lane, a.DP - 1 - 64 * (part % parts));
  const float *w = a.w + (int64_t)h * a.chunks * kChunk, *keep = a.keep + (int64_t)h * a.chunks;
  const bool live = d < a.DP;
  float n = a.pos > 0 ? a.n[(a.pos & 1) * slots + at] : 0.f;
  if (wave == 0 && live) a.nc[at] = n;
  float k[2][HALF], weight = 0.f, kept = 0.f;          // weight: that of token 4 (lane % 16) + lane / 16; kept: of 64 chunks
  auto chunk_of = [&](int c0) { return min(c0 + wave, a.chunks - 1); };
  auto request = [&](int c0, int half) {
    const int first = chunk_of(c0) * kChunk, last = min(first + kChunk, a.T) - 1;
#pragma unroll
    for (int i = 0; i < HALF; i++) k[half][i] = (rows + (int64_t)min(first + half * HALF + i, last) * a.ld_row)[column];
  };
  auto request_first = [&](int c0) {
    if ((c0 & 63) == 0) kept = keep[min(c0 + lane, a.chunks - 1)];
    weight = w[chunk_of(c0) * kChunk + lane];
    request(c0, 0);
  };
  request_first(0);
  for (int c0 = 0; c0 < a.chunks; c0 += WAVES, sums = c0 / WAVES & 1 ? sums + WAVES * 64 : sums - WAVES * 64) {
    const int count = a.T - chunk_of(c0) * kChunk;
    const float held = kept;
    request(c0, 1);
    float u = 0.f;
    {
#pragma clang fp contract(off)
#pragma unroll
      for (int t = 0; t < kChunk; t++)
        u = u + (t < count ? k[t / HALF][t % HALF] : 0.f) * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), 16 * (t & 3) + (t >> 2)));
    }
    if (c0 + WAVES < a.chunks) request_first(c0 + WAVES);
    sums[64 * wave + lane] = u;
    __syncthreads();                                   // (the other half of the sums is written next)
#pragma unroll
    for (int i = 0; i < WAVES; i++) {
      const int c = c0 + i;
      if (c >= a.chunks) break;
      n = fmaf(n, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(held), c & 63)), sums[64 * i + lane]);
      if (i == wave && live && c + 1 < a.chunks) a.nc[(c + 1) * slots + at] = n;
    }
  }
  if (wave == 0 && live) a.n[((a.pos + a.T) & 1) * slots + at] = n;
}

template <int ROWS>
__global__ __launch_bounds__(StateTile<ROWS>::kThreads, ROWS == 64 ? 4 : 2) void mlstm_states_kernel(const MemArgs a) {
  using Tile = StateTile<ROWS>;
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int tiles_v = a.VP / 32, per_head = (a.DP + ROWS - 1) / ROWS * tiles_v, tiles = per_head * a.H;
  if ((int)blockIdx.x >= tiles) {
    walk_normaliser<Tile::kWaves>(a, (int)blockIdx.x - tiles, reinterpret_cast<float*>(lds));
    return;
  }
  const int tile = dh::xcd_contiguous(blockIdx.x, tiles);
  const int h = tile / per_head, d0 = ROWS * (tile % per_head / tiles_v), v0 = 32 * (tile % per_head % tiles_v);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const float* keep = a.keep + (int64_t)h * a.chunks;

  // state rows of waves past the last: those 32 up, computed twice
  const int wd = d0 + 16 * (wave >> 1) < a.DP ? 16 * (wave >> 1) : 16 * (wave >> 1) - 32, wv = 16 * (wave & 1);
  const int64_t size = (int64_t)a.DP * a.VP;
  // accumulator element e of a lane: state row 4 (lane / 16) + e, column lane % 16
  const int64_t at = (int64_t)h * size + (int64_t)(d0 + wd + 4 * (lane >> 4)) * a.VP + v0 + wv + (lane & 15);
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  if (a.pos > 0) {
#pragma unroll
    for (int e = 0; e < 4; e++) s[e] = a.S[at + (int64_t)e * a.VP];
  }
  float* front = a.Sc + at;                            // in front of the next chunk
  auto store = [&](float* to) {
#pragma unroll
    for (int e = 0; e < 4; e++) to[(int64_t)e * a.VP] = s[e];
  };
  store(front);
  float kept = keep[min(lane, a.chunks - 1)];          // of 64 chunks
  asm volatile("" : "+v"(kept));                       // the compiler's own loads are over before fetches are counted

  // a wave's fetches of a chunk: its tokens' keys and values, and the weights (every wave the same); past the last chunk that again, unread
  const float* rows = a.rows + (int64_t)h * a.DP;
  auto key_token = [&](int r) { return Tile::kKeyTokens * (Tile::kKeyFetches * wave + r) + lane / Tile::kPieces; };
  auto value_token = [&](int r) { return 8 * (Tile::kValueFetches * wave + r) + (lane >> 3); };
  auto key_at = [&](int t) { return a.k_off + min(d0 + 4 * ((lane % Tile::kPieces) ^ Tile::key_swap(t)), a.DP - 4); };
  auto value_at = [&](int t) { return a.v_off + h * (a.VP - a.DP) + v0 + 4 * ((lane & 7) ^ Tile::value_swap(t)); };
  const float *key_from[Tile::kKeyFetches], *value_from[Tile::kValueFetches];
#pragma unroll
  for (int r = 0; r < Tile::kKeyFetches; r++) key_from[r] = rows + (int64_t)key_token(r) * a.ld_row + key_at(key_token(r));
#pragma unroll
  for (int r = 0; r < Tile::kValueFetches; r++) value_from[r] = rows + (int64_t)value_token(r) * a.ld_row + value_at(value_token(r));
  const float* weights_from = a.w + (int64_t)h * a.chunks * kChunk + lane;
  const int64_t chunk_step = (int64_t)kChunk * a.ld_row;
  int next = 0;                                        // the chunk to be fetched next
  uint32_t next_buf = lds0;
  auto fetch = [&](int i) {                            // the i-th of kFetches
    const bool tail = (next + 1) * kChunk >= a.T;      // the last chunk, or past it
    const int first = (a.chunks - 1) * kChunk, last = a.T - 1;
    if (i < Tile::kKeyFetches) {
      const int t = key_token(i);
      const float* from = key_from[i];
      if (tail) from = rows + (int64_t)min(first + t, last) * a.ld_row + key_at(t);
      dh::fetch_global_to_lds(from, next_buf + 1024 * (Tile::kKeyFetches * wave + i));
      key_from[i] += chunk_step;
    } else if (i < Tile::kKeyFetches + Tile::kValueFetches) {
      const int r = i - Tile::kKeyFetches, t = value_token(r);
      const float* from = value_from[r];
      if (tail) from = rows + (int64_t)min(first + t, last) * a.ld_row + value_at(t);
      dh::fetch_global_to_lds(from, next_buf + Tile::kKeys + 1024 * (Tile::kValueFetches * wave + r));
      value_from[r] += chunk_step;
    } else {
      dh::fetch_words_to_lds(weights_from, lds0 + Tile::kWeights + 4 * kChunk * (next & 3));
      if (!tail) weights_from += kChunk;
      next++;
      next_buf = next_buf == lds0 + (Tile::kBuffers - 1) * Tile::kBuffer ? lds0 : next_buf + Tile::kBuffer;
    }
  };
#pragma unroll
  for (int n = 0; n < 3; n++)
#pragma unroll
    for (int i = 0; i < Tile::kFetches; i++) fetch(i);
  // a lane's operands: token 4 j + tq, row wd + lane % 16 and column wv + lane % 16
  const int tq = lane >> 4, kd = wd + (lane & 15), vc = wv + (lane & 15);
  const uint32_t k_at = 4 * ROWS * tq + 16 * ((kd >> 2) ^ Tile::key_swap(tq)) + 4 * (kd & 3);
  const uint32_t v_at = Tile::kKeys + 128 * tq + 16 * ((vc >> 2) ^ Tile::value_swap(tq)) + 4 * (vc & 3);
  struct Operands {
    float k[kChunk / 4], v[kChunk / 4];
  };
  const char* buf = lds;
  auto read = [&](Operands& o, int j) {
    o.k[j] = *reinterpret_cast<const float*>(buf + k_at + 16 * ROWS * j);
    o.v[j] = *reinterpret_cast<const float*>(buf + v_at + 512 * j);
  };
  auto next_buffer = [&] { buf = buf == lds + (Tile::kBuffers - 1) * Tile::kBuffer ? lds : buf + Tile::kBuffer; };
  // a chunk is multiplied while the next one's operands are read and the third after it is fetched into the buffer it came from
  auto step = [&](int c, Operands& now, Operands& next) {
    // chunk c + 1 is there: younger than its fetches are those of c + 2 and the stores of the two chunks before this
    if (c >= 2) dh::arrive_and_wait<Tile::kFetches + 8>();
    else if (c == 1) dh::arrive_and_wait<Tile::kFetches + 4>();
    else dh::arrive_and_wait<Tile::kFetches>();
    const int count = a.T - c * kChunk;
#pragma unroll
    for (int j = 0; j < kChunk / 16; j++) {            // a quarter's weights lie side by side (mlstm_gates_kernel)
      const f32x4_t w = *reinterpret_cast<const f32x4_t*>(lds + Tile::kWeights + 4 * kChunk * (c & 3) + 64 * tq + 16 * j);
#pragma unroll
      for (int e = 0; e < 4; e++) now.k[4 * j + e] *= w[e];
    }
    if (count < kChunk) {                              // (rows past the last repeat it: an infinite one times a weight of zero is no number)
#pragma unroll
      for (int j = 0; j < kChunk / 4; j++)
        if (4 * j + tq >= count) now.k[j] = now.v[j] = 0.f;
    }
    f32x4_t u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kChunk / 4; j++) {
      u = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[j], now.v[j], u, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      read(next, j);
      if (j % 2 && j / 2 < Tile::kFetches) fetch(j / 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(Tile::kFetches <= kChunk / 8, "all of them in between");
    if ((c & 63) == 0 && c > 0) {
      kept = keep[min(c + lane, a.chunks - 1)];
      asm volatile("" : "+v"(kept));                   // waited for here, not at every chunk
    }
    const float left = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(kept), c & 63));
    s = s * left + u;
    front = c + 1 < a.chunks ? front + a.H * size : a.S + at;      // (nobody reads the state behind the last chunk from the workspace)
    store(front);
    next_buffer();
  };
  Operands even, odd;
  dh::arrive_and_wait<2 * Tile::kFetches>();
#pragma unroll
  for (int j = 0; j < kChunk / 4; j++) read(even, j);
  next_buffer();
  for (int c = 0; c < a.chunks; c += 2) {
    step(c, even, odd);
    if (c + 1 >= a.chunks) break;
    step(c + 1, odd, even);
  }
  dh::arrive_and_wait<0>();                            // nothing may be in flight towards LDS when the workgroup ends
}

// 2^y of a double, in f32: the whole part goes into the exponent, so that the f32 exponential sees at most a half.
__device__ __forceinline__ float exp2_of(double y) {
  const double whole = __builtin_rint(y);
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((float)(y - whole)), (int)whole);
}

// o of 64 tokens x 64 value columns of a (chunk, head): Q S over dim, decayed, plus the decayed and masked scores times V; four waves of 32 x 32.
// Grid: x = eight (chunk, head) pairs, one a die, under the column groups; y and z = eights of pairs.  So the column groups of a pair follow one
// another on a die, whose L2 then holds its rows and scores.
// Bound by the 32-bit matrix cores (160 instructions of 64 cycles a wave) and by what a step does besides: 64 dims' rows go through registers into LDS
// in front of each quarter of the products, requested by offsets that are computed once (address arithmetic at every step took as long as the products).
// us, four heads of 256 x 512, 1531 tokens (24 chunks: 768 workgroups, three a compute unit) 28 against 46.6 with Q K^T in here, once for each 128
// columns (384 workgroups of twice the columns), and exponentials by expf; 40 tokens, four heads of 128 x 256, 8.6 against 14.4.
// FAR: 64 rows span more than 4 GB.
template <bool FAR>
__global__ __launch_bounds__(256, 3) void mlstm_outputs_kernel(const MemArgs a) {
  using Offset = std::conditional_t<FAR, uint64_t, uint32_t>;
  // rows of LDS: read across rows (queries, scores) or across columns of rows four apart (states, values)
  constexpr int BD = 64, ROW = kScoreRow, VROW = 64 + 8;
  constexpr double kLog2e = 1.4426950408889634;
  __shared__ __align__(16) float qs[kChunk * ROW];
  __shared__ __align__(16) float sv[kChunk * VROW];
  __shared__ __align__(16) double decay_to[kChunk];    // a score's decay: 2^(to[t] + from[s])
  __shared__ __align__(16) double decay_from[kChunk];
  __shared__ float inter[kChunk];                      // what the state before the chunk has decayed to, per token
  __shared__ float least[kChunk];                      // e^-m
  __shared__ float factor[kChunk];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int group = blockIdx.x >> 3, ch = (blockIdx.x & 7) + 8 * (blockIdx.y + gridDim.y * blockIdx.z), v0 = 64 * group;
  if (ch >= a.chunks * a.H) return;
  const int c = ch / a.H, h = ch - c * a.H;
  const int first = c * kChunk, count = min(kChunk, a.T - first);
  // (the waves of the first 32 tokens have half of the scores: every other column group turns them round)
  const int wt = 32 * ((wave >> 1) ^ (group & 1)), wc = 32 * (wave & 1);
  // a thread's rows r0 + 16 r and its columns x .. x + 3 of every 64; offsets in bytes from bases all threads share
  const int r0 = tid >> 4, x = 4 * (tid & 15), v = min(v0 + x, a.VP - 4);
  const float *q_base = a.rows + (int64_t)first * a.ld_row + (int64_t)h * a.DP, *s_base = a.Sc + (int64_t)ch * a.DP * a.VP, *n_base = a.nc + (int64_t)ch * a.DP;
  Offset q_off[4];
#pragma unroll
  for (int r = 0; r < 4; r++) q_off[r] = 4 * ((Offset)min(r0 + 16 * r, count - 1) * (Offset)a.ld_row + x);
  const Offset s_off = 4 * ((Offset)r0 * a.VP + v);
  f32x4_t qr[4], sr[4], nr;
  auto at = [](const float* base, Offset off) { return *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const char*>(base) + off); };
  // (where dims are no multiple of 64 the last step reads up to 32 dims past them, of what follows in a row and in the workspace, and drops them)
  auto request = [&](int d0) {
#pragma unroll
    for (int r = 0; r < 4; r++) qr[r] = at(q_base + d0, q_off[r]);
#pragma unroll
    for (int r = 0; r < 4; r++) sr[r] = at(s_base + (int64_t)(d0 + 16 * r) * a.VP, s_off);
    nr = at(n_base + d0, 4 * x);
  };
  request(0);
  if (tid < kChunk) {
    const int t = first + min(tid, count - 1);
    const double F_start = first > 0 ? a.F[(int64_t)h * a.T + first - 1] : 0.0, F = a.F[(int64_t)h * a.T + t];
    const float m = a.mt[(int64_t)h * a.T + t];
    decay_to[tid] = (F - (double)m) * kLog2e;
    decay_from[tid] = ((double)a.i[(int64_t)h * a.T + t] - F) * kLog2e;
    inter[tid] = expf((float)(F - F_start + (double)a.mc[(int64_t)h * (a.chunks + 1) + c] - (double)m));
    least[tid] = expf(-m);
  }
  f32x16_t o;
#pragma unroll
  for (int e = 0; e < 16; e++) o[e] = 0.f;
  float dot[4] = {0.f, 0.f, 0.f, 0.f};                 // n_start . q of the thread's rows
  auto store = [&] {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      *reinterpret_cast<f32x4_t*>(&qs[(r0 + 16 * r) * ROW + x]) = qr[r];
      *reinterpret_cast<f32x4_t*>(&sv[(r0 + 16 * r) * VROW + x]) = sr[r];
    }
  };
  // o += rows of qs times columns of sv over so many eights of either; the next eight are read while these are multiplied
  auto multiply = [&](auto eights) {
    constexpr int N = decltype(eights)::value;
    f32x4_t fq[2], fs[2];
    auto read = [&](int s) {
      const int d = 8 * s + 4 * (lane >> 5);
      fq[s & 1] = *reinterpret_cast<const f32x4_t*>(&qs[(wt + (lane & 31)) * ROW + d]);
#pragma unroll
      for (int e = 0; e < 4; e++) fs[s & 1][e] = sv[(d + e) * VROW + wc + (lane & 31)];
    };
    read(0);
#pragma unroll
    for (int s = 0; s < N; s++) {
      if (s + 1 < N) read(s + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; e++) o = __builtin_amdgcn_mfma_f32_32x32x2f32(fq[s & 1][e], fs[s & 1][e], o, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int d0 = 0; d0 < a.DP; d0 += BD) {
    if (d0 + BD > a.DP) {                              // the upper half of these dims is not there (sizes are multiples of 32)
      if (x >= 32) {
        nr = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; r++) qr[r] = nr;
      }
      sr[2] = sr[3] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      qr[r] *= a.q_scale;
#pragma unroll
      for (int e = 0; e < 4; e++) dot[r] = fmaf(qr[r][e], nr[e], dot[r]);
    }
    __syncthreads();
    store();
    __syncthreads();
    // the next dims' rows, behind the last ones scores and values
    if (d0 + BD < a.DP) {
      request(d0 + BD);
    } else {
      const float *p_base = a.scores + (int64_t)ch * (kChunk * kChunk), *v_base = q_base + (a.v_off + (int64_t)h * (a.VP - a.DP) + v - x);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        qr[r] = at(p_base + 16 * kChunk * r, 16 * tid);
        sr[r] = at(v_base, q_off[r]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(std::integral_constant<int, BD / 8>{});
  }
  // decayed scores (nothing of what lies past the diagonal is a score), and with their sums the factor of a token's outputs
  double from[4];
#pragma unroll
  for (int e = 0; e < 4; e++) from[e] = decay_from[x + e];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int t = r0 + 16 * r;
    const double to = decay_to[t];
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float decayed = exp2_of(to + from[e]) * qr[r][e];
      qr[r][e] = x + e <= t && x + e < count ? decayed : 0.f;
      sum += qr[r][e];
    }
    sum = dh::group_combine<1, 16>(sum, dh::AddOp());
    const float nq = dh::group_combine<1, 16>(dot[r], dh::AddOp());
    if (x == 0) factor[t] = 1.0f / (fmaxf(fabsf(fmaf(inter[t], nq, sum)), least[t]) + kDenominatorEps);
    if (t >= count) sr[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  store();
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 16; e++) o[e] *= inter[wt + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)];
  if (__builtin_amdgcn_readfirstlane(wt)) multiply(std::integral_constant<int, kChunk / 8>{});
  else multiply(std::integral_constant<int, kChunk / 16>{});         // tokens 0 .. 31 have no scores past them
#pragma unroll
  for (int e = 0; e < 16; e++) o[e] *= factor[wt + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)];
  const int col = v0 + wc + (lane & 31);
  if (col >= a.VP) return;
  float* out = a.out + (int64_t)(first + wt + 4 * (lane >> 5)) * a.ld_out + (int64_t)h * a.VP + col;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int t = 8 * (e >> 2) + (e & 3);
    if (wt + 4 * (lane >> 5) + t < count) out[(int64_t)t * a.ld_out] = o[e];
  }
}

// One wave per (row, head): y = x / rms(x over size) * weight * sigmoid(gate).
template <typename OUT>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ x, int64_t ld_x, const float* __restrict__ gate,
                                                             int64_t ld_gate, const float* __restrict__ w, OUT* __restrict__ out,
                                                             int64_t ld_out, int rows, int H, int VP, int size, float eps) {
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), item = 4 * blockIdx.x + wave, row = item / (uint32_t)H;
  const int lane = threadIdx.x & 63, h = (int)(item - row * (uint32_t)H);
  if (row >= (uint32_t)rows) return;
  const int64_t t = row;
  const float* xr = x + t * ld_x + (int64_t)h * VP;
  float ss = 0.f;
  for (int i = 4 * lane; i < VP; i += 256) {
    const float4 v = *reinterpret_cast<const float4*>(xr + i);
    ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
  }
  ss = dh::wave_sum_uniform(ss);
  const float inv = 1.0f / sqrtf(ss / (float)size + eps);
  for (int i = 4 * lane; i < VP; i += 256) {
    const float4 v = *reinterpret_cast<const float4*>(xr + i);
    const float4 g = *reinterpret_cast<const float4*>(gate + t * ld_gate + (int64_t)h * VP + i);
    const float4 c = *reinterpret_cast<const float4*>(w + (int64_t)h * VP + i);
    const float y[4] = {v.x * inv * c.x / (1.0f + expf(-g.x)), v.y * inv * c.y / (1.0f + expf(-g.y)),
                        v.z * inv * c.z / (1.0f + expf(-g.z)), v.w * inv * c.w / (1.0f + expf(-g.w))};
    OUT* o = out + t * ld_out + (int64_t)h * VP + i;
    if constexpr (sizeof(OUT) == 2) {
      uint2 two;
      two.x = (uint32_t)dh::f32_to_bf16_bits(y[0]) | ((uint32_t)dh::f32_to_bf16_bits(y[1]) << 16);
      two.y = (uint32_t)dh::f32_to_bf16_bits(y[2]) | ((uint32_t)dh::f32_to_bf16_bits(y[3]) << 16);
      *reinterpret_cast<uint2*>(o) = two;
    } else {
      *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
    }
  }
}

int check(const char* op, const dh_mlstm* s) {
  if (!s) return dh::fail(1, "[%s] null spec", op);
  if (s->H <= 0 || s->dim <= 0 || s->vdim <= 0 || s->DP < s->dim || s->VP < s->vdim || s->DP % 32 || s->VP % 32)
    return dh::fail(1, "[%s] heads %d of %d x %d in padded sizes %d x %d (multiples of 32)", op, s->H, s->dim, s->vdim, s->DP, s->VP);
  if (!(s->gate_cap > 0.f)) return dh::fail(1, "[%s] the gate cap must be positive", op);
  const int64_t nq = (int64_t)s->H * s->DP, nv = (int64_t)s->H * s->VP;
  if ((s->ld_row | s->k_offset | s->v_offset) % 4 || s->k_offset < nq || s->v_offset < 0 || s->i_offset < 0 || s->f_offset < 0 ||
      s->ld_row < std::max<int64_t>(std::max<int64_t>(s->k_offset + nq, s->v_offset + nv), (int64_t)std::max(s->i_offset, s->f_offset) + s->H))
    return dh::fail(1, "[%s] a projection row of %d floats does not hold its parts", op, s->ld_row);
  return 0;
}
size_t up256(size_t n) { return (n + 255) / 256 * 256; }

MemArgs make_args(const dh_mlstm* s, const float* rows, float* state, float* out) {
  MemArgs a{};
  a.rows = rows; a.S = state; a.n = state + (size_t)s->H * s->DP * s->VP; a.m = a.n + (size_t)2 * s->H * s->DP; a.out = out;
  a.ld_row = s->ld_row; a.H = s->H; a.DP = s->DP; a.VP = s->VP;
  a.k_off = s->k_offset; a.v_off = s->v_offset; a.i_off = s->i_offset; a.f_off = s->f_offset;
  a.gate_cap = s->gate_cap; a.q_scale = 1.0f / sqrtf((float)s->dim);
  return a;
}
bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Rows of the states' tiles, 0: two launches.  Tiles of 64 rows, or of 32 where those would not fill the device (us, 64 / 32: 128 x 256 34 /
// 28.4, 256 x 512 36 / 41).  A walk takes 0.64 us a chunk however few its tiles are, two launches 0.22 where few and 0.65 where there are
// 32 of 64 x 64 (one workgroup a chunk each): us for state and chunks, walk / two launches: 1 x 64 x 64 (one tile) 1000 tokens 12.3 / 12.4, 2048 22 / 15.6,
// 8192 82 / 36; 2 x 128 x 256 (16 tiles) 1500 19 / 20.8, 8192 83 / 64; 4 x 128 x 256 (32) 2048 24.7 / 28.6, 8192 86 / 94.
int walk_rows(const dh_mlstm& s, int chunks) {
  const int64_t tiles = dh::ceil_div(s.DP, 64) * dh::ceil_div(s.VP, 64) * s.H;
  if (tiles < 32 && chunks > 16 + tiles / 2) return 0;
  return dh::ceil_div(s.DP, 64) * (s.VP / 32) * s.H >= dh::num_cus() ? 64 : 32;
}

template <int ROWS>
int launch_states(const char* op, const MemArgs& a) {
  using Tile = StateTile<ROWS>;
  auto kern = mlstm_states_kernel<ROWS>;
  static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::kBytes);
  DH_CHECK_HIP(op, set);
  hipLaunchKernelGGL(kern, dim3((unsigned)((dh::ceil_div(a.DP, ROWS) * (a.VP / 32) + dh::ceil_div(a.DP, 64)) * a.H)), dim3(Tile::kThreads), Tile::kBytes, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

}  // namespace

extern "C" {

size_t dh_mlstm_state_bytes(const dh_mlstm* s) {
  if (!s) return 0;
  return up256(((size_t)s->H * s->DP * s->VP + (size_t)2 * s->H * s->DP + (size_t)2 * s->H) * sizeof(float));
}

int dh_mlstm_step(const dh_mlstm* spec, const float* d_row, void* d_state, float* d_out, int pos, const uint32_t* d_kv_len) {
  const char* op = "dh_mlstm_step";
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, spec)) return rc;
  if (pos < 0) return dh::fail(1, "[%s] the position must be non-negative", op);
  if (!d_row || !d_state || !d_out) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_row) || !aligned(d_state) || !aligned(d_out)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  MemArgs a = make_args(spec, d_row, static_cast<float*>(d_state), d_out);
  a.pos = pos; a.kv_len = d_kv_len;
  hipLaunchKernelGGL(mlstm_step_kernel, dim3(spec->VP / kCols, spec->H), dim3(256), 0, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

size_t dh_mlstm_prefill_workspace_bytes(const dh_mlstm* s, int T) {
  if (!s || T <= 0) return 256;
  const size_t chunks = (size_t)dh::ceil_div(T, kChunk), HT = (size_t)s->H * T;
  return up256(HT * 8) + 2 * up256(HT * 4) + 2 * up256((size_t)s->H * (chunks + 1) * 4) + up256((size_t)s->H * chunks * kChunk * 4) +
         up256((size_t)s->H * chunks * kChunk * kChunk * 4) + up256((chunks + 1) * s->H * s->DP * 4) +
         up256((chunks + 1) * s->H * s->DP * s->VP * 4);
}

int dh_mlstm_prefill_layout(const dh_mlstm* spec, int T, int num_cus, int64_t* out1) {
  const char* op = "dh_mlstm_prefill_layout";
  if (int rc = check(op, spec)) return rc;
  if (!out1 || T <= 0) return dh::fail(1, "[%s] T=%d, or no place for the result", op, T);
  dh::plan_begin(num_cus > 0 ? num_cus : dh::ready() ? dh::num_cus() : 256);
  *out1 = walk_rows(*spec, (int)dh::ceil_div(T, kChunk));
  dh::plan_end();
  return 0;
}

int dh_mlstm_prefill(const dh_mlstm* spec, const float* d_rows, void* d_state, void* d_workspace, float* d_out, int ld_out, int T,
                     int start_pos) {
  const char* op = "dh_mlstm_prefill";
  DH_REQUIRE_INIT(op);
  if (int rc = check(op, spec)) return rc;
  if (T <= 0 || start_pos < 0) return dh::fail(1, "[%s] seqLen must be positive and startPos non-negative", op);
  if (ld_out < spec->H * spec->VP || ld_out % 4) return dh::fail(1, "[%s] ld_out=%d must be a multiple of 4 and hold %d elements", op, ld_out, spec->H * spec->VP);
  if (!d_rows || !d_state || !d_workspace || !d_out) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_rows) || !aligned(d_state) || !aligned(d_out) || !aligned(d_workspace)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  MemArgs a = make_args(spec, d_rows, static_cast<float*>(d_state), d_out);
  a.pos = start_pos; a.T = T; a.chunks = (int)dh::ceil_div(T, kChunk); a.ld_out = ld_out;
  char* w = static_cast<char*>(d_workspace);
  auto take = [&](size_t bytes) { char* p = w; w += up256(bytes); return p; };
  const size_t HT = (size_t)spec->H * T;
  a.F = reinterpret_cast<double*>(take(HT * 8));
  a.i = reinterpret_cast<float*>(take(HT * 4));
  a.mt = reinterpret_cast<float*>(take(HT * 4));
  a.mc = reinterpret_cast<float*>(take((size_t)spec->H * (a.chunks + 1) * 4));
  a.keep = reinterpret_cast<float*>(take((size_t)spec->H * (a.chunks + 1) * 4));
  a.w = reinterpret_cast<float*>(take((size_t)spec->H * a.chunks * kChunk * 4));
  a.scores = reinterpret_cast<float*>(take((size_t)spec->H * a.chunks * kChunk * kChunk * 4));
  a.nc = reinterpret_cast<float*>(take((size_t)(a.chunks + 1) * spec->H * spec->DP * 4));
  a.Sc = reinterpret_cast<float*>(take((size_t)(a.chunks + 1) * spec->H * spec->DP * spec->VP * 4));
  // (more chunks than a grid's smaller dimensions hold have always been refused)
  if (a.chunks > 65535) return dh::fail(1, "[%s] %d tokens are too many for one portion", op, T);
  const int rows = walk_rows(*spec, a.chunks);
  if (!rows) a.w = nullptr;
  hipLaunchKernelGGL(mlstm_gates_kernel, dim3(a.chunks + 1, spec->H), dim3(1024), 0, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  if (rows) {
    if (int rc = rows == 64 ? launch_states<64>(op, a) : launch_states<32>(op, a)) return rc;
  } else {
    const int tiles = (int)(dh::ceil_div(spec->DP, 64) * dh::ceil_div(spec->VP, 64));
    hipLaunchKernelGGL(mlstm_chunks_kernel, dim3(tiles, spec->H, a.chunks), dim3(256), 0, dh::stream(), a);
    DH_CHECK_LAUNCH(op);
    hipLaunchKernelGGL(mlstm_scan_kernel, dim3((unsigned)dh::ceil_div((int64_t)spec->DP * spec->VP + spec->DP, 1024), spec->H), dim3(256), 0, dh::stream(), a);
    DH_CHECK_LAUNCH(op);
  }
  const int64_t eights = dh::ceil_div((int64_t)a.chunks * spec->H, 8), deep = dh::ceil_div(eights, 65535);
  // (a row of the workspace's states, 64 of which are offsets too, is never longer than one of these)
  auto outputs = (int64_t)4 * kChunk * a.ld_row < (int64_t)1 << 32 ? mlstm_outputs_kernel<false> : mlstm_outputs_kernel<true>;
  hipLaunchKernelGGL(outputs, dim3(8 * (unsigned)dh::ceil_div(spec->VP, 64), (unsigned)dh::ceil_div(eights, deep), (unsigned)deep), dim3(256), 0,
                     dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}

int dh_head_norm_gate(const float* d_x, int ld_x, const float* d_gate, int ld_gate, const float* d_weight, void* d_out, int out_dtype,
                      int ld_out, int rows, int H, int padded, int size, float eps) {
  const char* op = "dh_head_norm_gate";
  DH_REQUIRE_INIT(op);
  if (rows <= 0 || H <= 0 || size <= 0 || padded < size || padded % 4) return dh::fail(1, "[%s] %d rows of %d heads of %d elements (padded to %d)", op, rows, H, size, padded);
  if ((ld_x | ld_gate | ld_out) % 4 || std::min(ld_x, std::min(ld_gate, ld_out)) < H * padded)
    return dh::fail(1, "[%s] row strides must be multiples of 4 and hold %d elements (%d, %d, %d)", op, H * padded, ld_x, ld_gate, ld_out);
  if (out_dtype != DH_BF16 && out_dtype != DH_F32) return dh::fail(1, "[%s] output must be bf16 or f32, got dtype %d", op, out_dtype);
  if (!d_x || !d_gate || !d_weight || !d_out) return dh::fail(1, "[%s] null pointer", op);
  if (!aligned(d_x) || !aligned(d_gate) || !aligned(d_weight) || !aligned(d_out)) return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  const dim3 grid((unsigned)dh::ceil_div((int64_t)rows * H, 4));
  if (out_dtype == DH_BF16)
    hipLaunchKernelGGL(head_norm_gate_kernel<uint16_t>, grid, dim3(256), 0, dh::stream(), d_x, ld_x, d_gate, ld_gate, d_weight,
                       static_cast<uint16_t*>(d_out), ld_out, rows, H, padded, size, eps);
  else
    hipLaunchKernelGGL(head_norm_gate_kernel<float>, grid, dim3(256), 0, dh::stream(), d_x, ld_x, d_gate, ld_gate, d_weight,
                       static_cast<float*>(d_out), ld_out, rows, H, padded, size, eps);
  DH_CHECK_LAUNCH(op);
  return 0;
}

}  // extern "C"
