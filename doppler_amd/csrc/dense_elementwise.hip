// Token embedding sums and row norms of the dense-weight decoders.
#include <algorithm>

#include "dense_device.h"

namespace {

struct EmbedArgs {
  const uint32_t* ids;
  const uint32_t* prev;
  const uint16_t* embed;
  const uint16_t* bigram;
  const uint16_t* pos;
  float* out;
  int64_t buckets, mul_prev, mul_cur;
  int vocab, max_positions, ld_out, hidden, start_pos;
  const uint32_t* kv_len;
  // ONE form: a token from the host, whose id, key count and the token before it go to `words` on the way
  uint32_t* words;
  uint32_t id, count, before;
  int64_t bigram_row;
};

// Grid = (tokens, slices of 2048 columns): eight columns per thread with 16-byte loads where the rows are aligned for
// them, else one column at a time.  Rows that do not exist (id or position out of range) count as zeros, so no id read on
// the device can send a load outside the tables.
__host__ __device__ inline int64_t bigram_row(uint32_t prev, uint32_t cur, int64_t mul_prev, int64_t mul_cur, int64_t buckets) {
  const int64_t row = (int64_t)((uint64_t)(int64_t)prev * (uint64_t)mul_prev + (uint64_t)(int64_t)cur * (uint64_t)mul_cur) % buckets;
  return row < 0 ? row + buckets : row;
}
template <bool VEC, bool ONE>
__global__ __launch_bounds__(256) void embed_sum_kernel(const EmbedArgs a) {
  const int t = blockIdx.x;
  const int64_t p = !ONE && a.kv_len ? (int64_t)*a.kv_len - 1 : (int64_t)a.start_pos + t;
  const uint32_t id = ONE ? a.id : a.ids[t];
  if (ONE && blockIdx.y == 0 && threadIdx.x < 3) a.words[threadIdx.x] = threadIdx.x == 0 ? a.id : threadIdx.x == 1 ? a.count : a.before;
  const uint16_t* e = id < (uint32_t)a.vocab ? a.embed + (int64_t)id * a.hidden : nullptr;
  const uint16_t* b = nullptr;
  if (a.bigram) {
    int64_t row = ONE ? a.bigram_row : a.buckets;
    if (!ONE && p > 0) row = bigram_row(t > 0 ? a.ids[t - 1] : *a.prev, id, a.mul_prev, a.mul_cur, a.buckets);
    b = a.bigram + row * a.hidden;
  }
  const uint16_t* q = a.pos && p >= 0 && p < a.max_positions ? a.pos + p * a.hidden : nullptr;
  float* o = a.out + (int64_t)t * a.ld_out;
  const int first = 2048 * blockIdx.y;
  if (VEC) {
    const int i = first + 8 * threadIdx.x;
    if (i >= a.hidden) return;
    const dh::u32x4_t none = {0u, 0u, 0u, 0u};
    const dh::u32x4_t ev = e ? *reinterpret_cast<const dh::u32x4_t*>(e + i) : none;
    const dh::u32x4_t bv = b ? *reinterpret_cast<const dh::u32x4_t*>(b + i) : none;
    const dh::u32x4_t qv = q ? *reinterpret_cast<const dh::u32x4_t*>(q + i) : none;
    float v[8];
#pragma unroll
    for (int w = 0; w < 4; w++) {
      v[2 * w] = dh::bf16_low(ev[w]) + dh::bf16_low(bv[w]) + dh::bf16_low(qv[w]);
      v[2 * w + 1] = dh::bf16_high(ev[w]) + dh::bf16_high(bv[w]) + dh::bf16_high(qv[w]);
    }
    reinterpret_cast<float4*>(o + i)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(o + i)[1] = make_float4(v[4], v[5], v[6], v[7]);
    return;
  }
  const int last = min(first + 2048, a.hidden);
  for (int i = first + threadIdx.x; i < last; i += 256) {
    float v = e ? dh::bf16_bits_to_f32(e[i]) : 0.f;
    if (b) v += dh::bf16_bits_to_f32(b[i]);
    if (q) v += dh::bf16_bits_to_f32(q[i]);
    o[i] = v;
  }
}

// One workgroup per output row; the row stays in registers between the two passes (up to 8 x 1024 elements).
template <bool BF16>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* __restrict__ x, int ld_x, const uint32_t* rows,
                                                           const float* __restrict__ w, void* __restrict__ out, int ld_out,
                                                           int hidden, float eps) {
  __shared__ float red[4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const float* xr = x + (int64_t)(rows ? rows[blockIdx.x] : blockIdx.x) * ld_x;
  const int64_t base = (int64_t)blockIdx.x * ld_out;
  if ((ld_x & 3) == 0 && (hidden & 3) == 0 && hidden <= 1024 * dh::kNormPieces) {
    float4 xv[dh::kNormPieces];
#pragma unroll
    for (int j = 0; j < dh::kNormPieces; j++) {
      const int i = 4 * (tid + 256 * j);
      xv[j] = i < hidden ? *reinterpret_cast<const float4*>(xr + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    dh::store_normed_row<BF16>(xv, hidden, w, eps, red, out, base, ld_out);
    return;
  }
  float ss = 0.f;
  for (int i = tid; i < hidden; i += 256) ss = fmaf(xr[i], xr[i], ss);
  ss = dh::wave_sum_uniform(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)hidden + eps);
  auto put = [&](int i, float v) {
    if (BF16) static_cast<uint16_t*>(out)[base + i] = dh::f32_to_bf16_bits(v);
    else static_cast<float*>(out)[base + i] = v;
  };
  for (int i = tid; i < hidden; i += 256) put(i, xr[i] * inv * w[i]);
  for (int i = hidden + tid; i < ld_out; i += 256) put(i, 0.f);
}

}  // namespace

extern "C" {

static int embed_sum(const char* op, EmbedArgs a, int T, bool one) {
  DH_REQUIRE_INIT(op);
  if (T <= 0 || a.hidden <= 0 || a.vocab <= 0) return dh::fail(1, "[%s] Dimensions must be positive: T=%d, hidden=%d, vocab=%d", op, T, a.hidden, a.vocab);
  if (a.start_pos < 0) return dh::fail(1, "[%s] indexOffset and startPos must be non-negative", op);
  if (a.ld_out < a.hidden) return dh::fail(1, "[%s] ld_out=%d is shorter than hidden=%d", op, a.ld_out, a.hidden);
  if (!(one ? (const void*)a.words : a.ids) || !a.embed || !a.out) return dh::fail(1, "[%s] null pointer", op);
  if (a.kv_len && T != 1) return dh::fail(1, "[%s] the device key count serves one token, got T=%d", op, T);
  if (a.bigram && a.buckets <= 0) return dh::fail(1, "[%s] buckets must be positive", op);
  if (!one && a.bigram && !a.prev && (a.start_pos > 0 || a.kv_len)) return dh::fail(1, "[%s] the token before position %d is needed", op, a.start_pos);
  if (a.pos && (a.max_positions <= 0 || (!a.kv_len && a.start_pos + T > a.max_positions)))
    return dh::fail(1, "[%s] positions %d..%d are outside the table of %d", op, a.start_pos, a.start_pos + T - 1, a.max_positions);
  if (one && a.bigram) a.bigram_row = a.start_pos > 0 ? bigram_row(a.before, a.id, a.mul_prev, a.mul_cur, a.buckets) : a.buckets;
  const bool vec = a.hidden % 8 == 0 && a.ld_out % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(a.embed) | reinterpret_cast<uintptr_t>(a.bigram) | reinterpret_cast<uintptr_t>(a.pos) |
                     reinterpret_cast<uintptr_t>(a.out)) & 15) == 0;
  auto kern = vec ? one ? embed_sum_kernel<true, true> : embed_sum_kernel<true, false> : one ? embed_sum_kernel<false, true> : embed_sum_kernel<false, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)T, (unsigned)dh::ceil_div(a.hidden, 2048)), dim3(256), 0, dh::stream(), a);
  DH_CHECK_LAUNCH(op);
  return 0;
}
static EmbedArgs embed_args(const void* d_embed, int vocab, const void* d_bigram, int64_t buckets, int64_t mul_prev, int64_t mul_cur, const void* d_pos,
                            int max_positions, float* d_out, int ld_out, int hidden, int start_pos) {
  EmbedArgs a{};
  a.embed = static_cast<const uint16_t*>(d_embed); a.bigram = static_cast<const uint16_t*>(d_bigram);
  a.pos = static_cast<const uint16_t*>(d_pos);
  a.out = d_out; a.buckets = buckets; a.mul_prev = mul_prev; a.mul_cur = mul_cur;
  a.vocab = vocab; a.max_positions = max_positions; a.ld_out = ld_out; a.hidden = hidden; a.start_pos = start_pos;
  return a;
}

int dh_embed_sum(const uint32_t* d_ids, int index_offset, const uint32_t* d_prev, const void* d_embed, int vocab,
                 const void* d_bigram, int64_t buckets, int64_t mul_prev, int64_t mul_cur, const void* d_pos,
                 int max_positions, float* d_out, int ld_out, int T, int hidden, int start_pos, const uint32_t* d_kv_len) {
  EmbedArgs a = embed_args(d_embed, vocab, d_bigram, buckets, mul_prev, mul_cur, d_pos, max_positions, d_out, ld_out, hidden, index_offset < 0 ? -1 : start_pos);
  a.ids = d_ids ? d_ids + std::max(0, index_offset) : nullptr; a.prev = d_prev; a.kv_len = d_kv_len;
  return embed_sum("dh_embed_sum", a, T, false);
}

int dh_embed_sum_words(uint32_t* d_words, uint32_t id, uint32_t kv_len, uint32_t before, const void* d_embed, int vocab, const void* d_bigram, int64_t buckets,
                       int64_t mul_prev, int64_t mul_cur, const void* d_pos, int max_positions, float* d_out, int ld_out, int hidden, int pos) {
  EmbedArgs a = embed_args(d_embed, vocab, d_bigram, buckets, mul_prev, mul_cur, d_pos, max_positions, d_out, ld_out, hidden, pos);
  a.words = d_words; a.id = id; a.count = kv_len; a.before = before;
  DH_REQUIRE_INIT("dh_embed_sum_words");
  if (dh::capturing_graph()) return dh::fail(1, "[dh_embed_sum_words] not possible while a graph is being captured (a replay would set the same words)");
  return embed_sum("dh_embed_sum_words", a, 1, true);
}

int dh_rmsnorm_rows(const float* d_x, int ld_x, const uint32_t* d_rows, const float* d_weight, void* d_out, int out_dtype,
                    int ld_out, int n, int hidden, float eps) {
  const char* op = "dh_rmsnorm_rows";
  DH_REQUIRE_INIT(op);
  if (n <= 0 || hidden <= 0) return dh::fail(1, "[%s] Dimensions must be positive: rows=%d, hidden=%d", op, n, hidden);
  if (ld_x < hidden || ld_out < hidden) return dh::fail(1, "[%s] row strides must hold hidden=%d elements (%d, %d)", op, hidden, ld_x, ld_out);
  if (out_dtype != DH_BF16 && out_dtype != DH_F32) return dh::fail(1, "[%s] output must be bf16 or f32, got dtype %d", op, out_dtype);
  if (!d_x || !d_weight || !d_out) return dh::fail(1, "[%s] null pointer", op);
  if ((reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_weight) | reinterpret_cast<uintptr_t>(d_out)) & 15)
    return dh::fail(1, "[%s] pointers must be 16-byte aligned", op);
  if (out_dtype == DH_BF16)
    hipLaunchKernelGGL(rmsnorm_rows_kernel<true>, dim3(n), dim3(256), 0, dh::stream(), d_x, ld_x, d_rows, d_weight, d_out, ld_out, hidden, eps);
  else
    hipLaunchKernelGGL(rmsnorm_rows_kernel<false>, dim3(n), dim3(256), 0, dh::stream(), d_x, ld_x, d_rows, d_weight, d_out, ld_out, hidden, eps);
  DH_CHECK_LAUNCH(op);
  return 0;
}

}  // extern "C"
