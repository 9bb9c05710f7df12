// Device helpers of the dense (bf16-weight) kernels: element conversions, activations, lane reductions.
#pragma once
#include "dh_common.h"

namespace dh {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// A 32-bit word holds elements 2 i (low half) and 2 i + 1 (high half) of a bf16 row.
__device__ __forceinline__ float bf16_low(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_high(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float v) {      // round to nearest even
  return __builtin_bit_cast(uint16_t, (__bf16)v);
}

// DH_ACT_* of one value (a plain activation, not a gated pair); DH_ACT_NONE passes it through.
__device__ __forceinline__ float activate(float z, int act) {
  if (act == DH_ACT_RELU2) {
    const float r = fmaxf(z, 0.f);
    return r * r;
  }
  if (act == DH_ACT_SILU) return z / (1.0f + __expf(-z));
  if (act == DH_ACT_GELU) return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  if (act == DH_ACT_GELU_ERF) return 0.5f * z * (1.0f + erff(0.7071067811865476f * z));
  return z;
}

// A lane's value combined over aligned groups of SPAN lanes (2, 4, .. 64); every lane of the group ends with the
// result.  Steps inside a 16-lane row are DPP modifiers (quad permutations, then mirrors, which cross the halves
// of a group whose halves are already uniform), the last two the gfx950 lane-swap instructions: no LDS traffic.
template <int CTRL>
__device__ __forceinline__ float dpp_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xF, 0xF, false));
}
struct AddOp {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct MaxOp {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
// FROM < 64, TO <= 64: the group of TO lanes from groups of FROM lanes that are uniform already.
template <int FROM, int TO, typename Op>
__device__ __forceinline__ float group_combine(float v, Op op) {
  if (FROM < 2 && TO >= 2) v = op(v, dpp_lane<0xB1>(v));        // quad_perm 1,0,3,2
  if (FROM < 4 && TO >= 4) v = op(v, dpp_lane<0x4E>(v));        // quad_perm 2,3,0,1
  if (FROM < 8 && TO >= 8) v = op(v, dpp_lane<0x141>(v));       // row_half_mirror
  if (FROM < 16 && TO >= 16) v = op(v, dpp_lane<0x140>(v));     // row_mirror
  if (FROM < 32 && TO >= 32) {
    auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(s[0]), __uint_as_float(s[1]));
  }
  if (FROM < 64 && TO >= 64) {
    auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(s[0]), __uint_as_float(s[1]));
  }
  return v;
}

// A row that 256 threads hold, four elements at 4 (tid + 256 j) each (zeros past `hidden`, a multiple of 4 and at most 1024 PIECES), over its root mean square and
// times w, in the operand type of the product that reads it; columns hidden .. ld_out - 1 zero.
constexpr int kNormPieces = 8;
// Pieces where a row is made of several in the same launch.  Longer rows take a wide launch and the norm's: one workgroup's trips through 8192 columns of a few
// rows took longer than the launch they saved (products in slices with their norm, us, apart / in one, from 8192 columns: 16 x 4096 19.3 / 18.1, 5 x 5120
// 21.3 / 23.0, 16 x 6144 24.2 / 25.5, 33 x 8192 32.1 / 33.4; from 4096 200 x 7168 33.2 / 32.8).
constexpr int kMadePieces = 4;
template <bool BF16, int PIECES>
__device__ __forceinline__ void store_normed_row(const float4 (&xv)[PIECES], int hidden, const float* __restrict__ w, float eps, float* red, void* __restrict__ out,
                                                 int64_t base, int ld_out) {
  const int tid = threadIdx.x;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < PIECES; j++) {
    ss = fmaf(xv[j].x, xv[j].x, ss); ss = fmaf(xv[j].y, xv[j].y, ss);
    ss = fmaf(xv[j].z, xv[j].z, ss); ss = fmaf(xv[j].w, xv[j].w, ss);
  }
  ss = wave_sum_uniform(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)hidden + eps);
  auto put = [&](int i, float v) {
    if (BF16) static_cast<uint16_t*>(out)[base + i] = f32_to_bf16_bits(v);
    else static_cast<float*>(out)[base + i] = v;
  };
#pragma unroll
  for (int j = 0; j < PIECES; j++) {
    const int i = 4 * (tid + 256 * j);
    if (i >= hidden) continue;
    const float4 wv = *reinterpret_cast<const float4*>(w + i);
    const float y[4] = {xv[j].x * inv * wv.x, xv[j].y * inv * wv.y, xv[j].z * inv * wv.z, xv[j].w * inv * wv.w};
    if (BF16 && (ld_out & 3) == 0) {
      uint2 two;
      two.x = (uint32_t)f32_to_bf16_bits(y[0]) | ((uint32_t)f32_to_bf16_bits(y[1]) << 16);
      two.y = (uint32_t)f32_to_bf16_bits(y[2]) | ((uint32_t)f32_to_bf16_bits(y[3]) << 16);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + base + i) = two;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) put(i + e, y[e]);
    }
  }
  for (int i = hidden + tid; i < ld_out; i += 256) put(i, 0.f);
}

// Workgroup index -> tile index such that each of the eight XCDs (which the hardware deals workgroups to in turn)
// gets a contiguous run of tiles and its L2 sees their shared operands.
__device__ __forceinline__ int xcd_contiguous(int id, int total) {
  const int xcd = id & 7, within = id >> 3, q = total >> 3, r = total & 7;
  return xcd * q + (xcd < r ? xcd : r) + within;
}

}  // namespace dh
