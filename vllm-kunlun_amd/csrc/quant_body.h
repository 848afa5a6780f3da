// Per-row dynamic int8 and per-group fp8 quantisation as device functions, shared by the stand-alone
// kernels and the fused routing + quantisation launch.
#pragma once
#include "kmoe_common.h"

namespace kmoe {

union Pack8 {  // 8 bf16 (or half) values
  uint4 v;
  uint16_t h[8];
};

// ---------------------------------------------------------------- int8 rows
// TPR threads cooperate on one row (32: two rows per wave); each keeps NV vectors of 8 values in
// registers, so the row is read from memory once.
// Workgroup `block` (256 threads) serves rows block * (256 / TPR) ...
template <int TPR, int NV>
__device__ inline void quant_i8_rows_body(const uint16_t* __restrict__ x, int64_t ld_x, int R, int C,
                                          int8_t* __restrict__ q, int64_t ld_q, float* __restrict__ row_max,
                                          int chunked, int block, bool f16 = false) {
  constexpr int kRowsPerBlock = 256 / TPR;
  __shared__ float red[256 / kWave];
  const int sub = threadIdx.x / TPR;
  const int t = threadIdx.x % TPR;
  const int r = block * kRowsPerBlock + sub;
  const bool live = r < R;
  const int nvec = C / 8;
  Pack8 val[NV];
  float amax = 0.0f;
  if (live) {
    const uint4* src = reinterpret_cast<const uint4*>(x + static_cast<size_t>(r) * ld_x);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = t + i * TPR;
      if (v < nvec) {
        val[i].v = src[v];
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(act_to_f32(val[i].h[j], f16)));
      }
    }
  }
  amax = group_max<(TPR < kWave ? TPR : kWave)>(amax);
  if (TPR > kWave) {  // one row per block: combine the waves
    if (lane_id() == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < TPR / kWave; ++w) amax = fmaxf(amax, red[w]);
  }
  if (!live) return;
  const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
  // row-major: vector v of the row; chunk-major [C/64][R][64]: vector v is eighth v%8 of chunk v/8
  uint2* dst = reinterpret_cast<uint2*>(q + static_cast<size_t>(r) * (chunked ? 64 : ld_q));
  const size_t vstride = chunked ? static_cast<size_t>(R) : 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = t + i * TPR;
    if (v < nvec) {
      uint32_t w[2] = {0, 0};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = __builtin_rintf(act_to_f32(val[i].h[j], f16) * inv);
        f = fminf(fmaxf(f, -127.0f), 127.0f);
        const int qi = static_cast<int>(f);
        w[j >> 2] |= static_cast<uint32_t>(qi & 0xff) << (8 * (j & 3));
      }
      dst[chunked ? (v >> 3) * vstride * 8 + (v & 7) : v] = make_uint2(w[0], w[1]);
    }
  }
  if (t == 0) row_max[r] = amax;
}

// ------------------------------------------------------------- fp8 group128
// OCP e4m3fn encode of two floats, round-to-nearest-even, saturating at 448 (NaN -> the largest
// code of its sign): the conversion instruction of gfx950 (v_cvt_pk_fp8_f32 encodes the OCP format
// there) after an explicit clamp, so that its own overflow handling never comes into play.
__device__ inline uint32_t pack2_e4m3fn(float a, float b) {
  auto clamp = [](float f) {
    f = f != f ? __builtin_copysignf(448.0f, f) : f;
    return __builtin_fminf(__builtin_fmaxf(f, -448.0f), 448.0f);
  };
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(clamp(a), clamp(b), 0, false)) & 0xffffu;
}

// 16 lanes x 8 values = one 128-column group; 4 groups per wave. Bound by instruction issue before it is by memory (eight
// IEEE divisions, clamps and NaN tests per lane took 62 us for [27009, 2048], 2.7 TB/s; this takes 39, 4.3 TB/s), so: the largest magnitude by integer
// maxima of the 16-bit patterns, two per instruction (a NaN shows as one above infinity), and x / s from the rounded
// reciprocal y = 1 / s by one step of Markstein's division, q = x y, q + (x - q s) y with fused steps. That is the
// correctly rounded quotient for every 8- and 11-bit mantissa of x and of the group's maximum (s is the maximum over
// 448; all combinations were compared, down to x = 2^-24 of the maximum), as long as neither s nor 1 / s nor the remainder
// leaves the normal range: other groups, and those with a NaN, divide. No value beyond 448 reaches the conversion by more
// than the quotient's rounding, so the quick way needs no clamp.
__device__ inline void quant_fp8_group128_body(const uint16_t* __restrict__ x, int64_t ld_x, int R, int C,
                                               uint8_t* __restrict__ q, int64_t ld_q, float* __restrict__ scale,
                                               int block, bool f16) {
  typedef unsigned short v2us __attribute__((ext_vector_type(2)));
  const int groups_per_row = C / 128;
  const long long total = static_cast<long long>(R) * groups_per_row;
  const long long gid = static_cast<long long>(block) * 16 + (threadIdx.x >> 4);
  const int t = threadIdx.x & 15;
  if (gid >= total) return;  // (a group's 16 lanes leave together)
  const int r = static_cast<int>(gid / groups_per_row);
  const int g = static_cast<int>(gid - static_cast<long long>(r) * groups_per_row);
  Pack8 val;
  val.v = *reinterpret_cast<const uint4*>(x + static_cast<size_t>(r) * ld_x + g * 128 + t * 8);
  auto magnitudes = [](uint32_t w) { return __builtin_bit_cast(v2us, w & 0x7fff7fffu); };
  const uint32_t m2 = __builtin_bit_cast(
      uint32_t, __builtin_elementwise_max(__builtin_elementwise_max(magnitudes(val.v.x), magnitudes(val.v.y)),
                                          __builtin_elementwise_max(magnitudes(val.v.z), magnitudes(val.v.w))));
  uint32_t m = max(m2 & 0xffffu, m2 >> 16);
  // maxima over the row of 16 lanes, rotated by 8, 4, 2 and 1
  m = max(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), 0x128, 0xf, 0xf, true)));
  m = max(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), 0x124, 0xf, 0xf, true)));
  m = max(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), 0x122, 0xf, 0xf, true)));
  m = max(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), 0x121, 0xf, 0xf, true)));
  float s = act_to_f32(static_cast<uint16_t>(m), f16) / 448.0f;
  uint32_t w[2] = {0, 0};
  if (s >= 0x1p-60f && s <= 0x1p60f) {  // (false for a NaN)
    const float y = 1.0f / s;
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = act_to_f32(val.h[j], f16);
      const float quotient = v * y;
      f[j] = __builtin_fmaf(-__builtin_fmaf(quotient, s, -v), y, quotient);  // (these signs keep a -0)
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int low = __builtin_amdgcn_cvt_pk_fp8_f32(f[4 * j], f[4 * j + 1], 0, false);
      w[j] = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(f[4 * j + 2], f[4 * j + 3], low, true));
    }
  } else {
    float amax = 0.0f;  // of the values that are numbers
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(act_to_f32(val.h[j], f16)));
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
    s = amax / 448.0f;
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = s > 0.0f ? act_to_f32(val.h[j], f16) / s : 0.0f;
    w[0] = pack2_e4m3fn(f[0], f[1]) | (pack2_e4m3fn(f[2], f[3]) << 16);
    w[1] = pack2_e4m3fn(f[4], f[5]) | (pack2_e4m3fn(f[6], f[7]) << 16);
  }
  *reinterpret_cast<uint2*>(q + static_cast<size_t>(r) * ld_q + g * 128 + t * 8) = make_uint2(w[0], w[1]);
  if (t == 0) scale[static_cast<size_t>(r) * groups_per_row + g] = s;
}

}  // namespace kmoe
