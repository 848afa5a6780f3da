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
// What the quantisers share. The largest magnitude of a row is found on the 16-bit patterns, two per instruction: without
// the sign they are ordered as the numbers are, infinities above every number and NaNs above those.
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
__device__ inline uint32_t max_magnitudes(uint32_t a, uint32_t b) {  // of two pairs of magnitudes
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2us, a), __builtin_bit_cast(v2us, b)));
}
__device__ inline uint32_t magnitudes8(const Pack8& v) {
  return max_magnitudes(max_magnitudes(v.v.x & 0x7fff7fffu, v.v.y & 0x7fff7fffu), max_magnitudes(v.v.z & 0x7fff7fffu, v.v.w & 0x7fff7fffu));
}
__device__ inline uint32_t max_of_pair(uint32_t m) { return max(m & 0xffffu, m >> 16); }

// The codes of 8 values, round(x * inv) with halves to even, inv = 127 / amax.
// quant8_i8: any values (clamped; a NaN gives -127). quant8_i8_number: all of them numbers and inv finite - then no
// product leaves [-127.5, 127.5], and adding 1.5 * 2^23 rounds it to an integer whose code is the sum's lowest byte: five
// instructions a value in place of twelve. The quantiser's launches were bound by them rather than by memory: [65536, 768]
// 32 -> 26 us (5.9 TB/s), [36864, 2048] 49 -> 41 us (5.5 TB/s).
__device__ inline uint2 quant8_i8(const Pack8& v, float inv, bool f16) {
  uint32_t w[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float f = __builtin_rintf(act_to_f32(v.h[j], f16) * inv);
    f = fminf(fmaxf(f, -127.0f), 127.0f);
    w[j >> 2] |= static_cast<uint32_t>(static_cast<int>(f) & 0xff) << (8 * (j & 3));
  }
  return make_uint2(w[0], w[1]);
}
template <bool F16>
__device__ inline uint2 quant8_i8_number(const Pack8& v, float inv) {
  uint32_t c[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    c[j] = __builtin_bit_cast(uint32_t, (F16 ? half_to_f32(v.h[j]) : bf16_to_f32(v.h[j])) * inv + 0x1.8p23f);
  // bytes, lowest first: of c[0], c[1], c[2], c[3]
  auto four = [&](int j) {
    const uint32_t lo = __builtin_amdgcn_perm(c[j + 1], c[j], 0x0c0c0400u), hi = __builtin_amdgcn_perm(c[j + 3], c[j + 2], 0x04000c0cu);
    return lo | hi;
  };
  return make_uint2(four(0), four(4));
}

// 127 / amax of a row whose largest magnitude has the pattern m, and whether quant8_i8_number may be used with it.
struct RowScale {
  float amax, inv;
  bool numbers;
};
__device__ inline RowScale row_scale_i8(uint32_t m, bool f16) {
  RowScale r;
  r.amax = act_to_f32(static_cast<uint16_t>(m), f16);
  r.inv = r.amax > 0.0f ? 127.0f / r.amax : 0.0f;
  r.numbers = m < (f16 ? 0x7c00u : 0x7f80u) && r.inv < __builtin_inff();
  return r;
}
__device__ inline uint2 quant8_i8_of(const Pack8& v, const RowScale& s, bool f16) {
  if (!s.numbers) return quant8_i8(v, s.inv, f16);
  return f16 ? quant8_i8_number<true>(v, s.inv) : quant8_i8_number<false>(v, s.inv);
}
// The largest magnitude of those values that are numbers or infinite: what a row with a NaN is scaled by.
__device__ inline float amax8(const Pack8& v, bool f16) {
  float m = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(act_to_f32(v.h[j], f16)));
  return m;
}

// TPR threads cooperate on one row (32: two rows per wave); each keeps NV vectors of 8 values in
// registers, so the row is read from memory once. A workgroup of THREADS serves rows first_row ..., or the one row first_row
// where that is a row's threads, more than a wave. Few rows are bound by
// the trip to memory: lanes past the row's end read its last vector again (which changes no maximum), because loads under
// conditions of their own went out one after another, each waiting for the one before. [64, 7168] 3.7 -> 2.8 us, [8, 2048]
// 3.3 -> 2.3, [4096, 7168] 16.8 -> 15.1, [8192, 768] 8.7 -> 7.9 (behind a launch that writes the rows).
// IN_TURN: each vector of a lane is waited for before the next is asked for.
template <int TPR, int NV, int THREADS = 256, bool IN_TURN = false>
__device__ __forceinline__ void quant_i8_rows_body(const uint16_t* __restrict__ x, int64_t ld_x, int R, int C,
                                                   int8_t* __restrict__ q, int64_t ld_q, float* __restrict__ row_max,
                                                   int chunked, uint32_t first_row, bool f16 = false) {
  static_assert(TPR <= kWave || TPR == THREADS, "rows of several waves have a workgroup each");
  __shared__ uint32_t red[THREADS / kWave];
  const int t = threadIdx.x % TPR;
  const uint32_t r = first_row + threadIdx.x / TPR;  // (a workgroup's last rows may lie beyond 2^31)
  const bool live = r < static_cast<uint32_t>(R);
  const int nvec = C / 8;
  Pack8 val[NV];
  const uint4* src = reinterpret_cast<const uint4*>(x + static_cast<size_t>(live ? r : static_cast<uint32_t>(R) - 1) * ld_x);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    val[i].v = src[min(t + i * TPR, nvec - 1)];
    if (IN_TURN && i + 1 < NV) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  }
  uint32_t mag = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) mag = max_magnitudes(mag, magnitudes8(val[i]));
  // max over the row's threads (one row per workgroup: combine the waves)
  auto row_max_of = [&](uint32_t m) {
    m = group_max_u32<(TPR < kWave ? TPR : kWave)>(m);
    if (TPR > kWave) {
      if (lane_id() == 0) red[threadIdx.x >> 6] = m;
      __syncthreads();
      m = red[0];
#pragma unroll
      for (int w = 1; w < TPR / kWave; ++w) m = max(m, red[w]);
    }
    return m;
  };
  RowScale s = row_scale_i8(row_max_of(max_of_pair(mag)), f16);
  if (!s.numbers) {  // (the same for all of a row's threads)
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) m = fmaxf(m, amax8(val[i], f16));
    if (TPR > kWave) __syncthreads();  // (every wave has read the maxima it is about to replace)
    s.amax = __builtin_bit_cast(float, row_max_of(__builtin_bit_cast(uint32_t, m)));  // (no negative numbers: ordered as their bits)
    s.inv = s.amax > 0.0f ? 127.0f / s.amax : 0.0f;
  }
  if (!live) return;
  // row-major: vector v of the row; chunk-major [C/64][R][64]: vector v is eighth v%8 of chunk v/8
  uint2* dst = reinterpret_cast<uint2*>(q + static_cast<size_t>(r) * (chunked ? 64 : ld_q));
  const size_t vstride = chunked ? static_cast<size_t>(R) : 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = t + i * TPR;
    if (v < nvec) {
      dst[chunked ? (v >> 3) * vstride * 8 + (v & 7) : v] = quant8_i8_of(val[i], s, f16);
    }
  }
  if (t == 0) row_max[r] = s.amax;
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
// quant8_fp8: the codes of this lane's 8 values of a group (the group's 16 lanes call together), its scale in `s`.
__device__ inline uint2 quant8_fp8(const Pack8& val, bool f16, float& s) {
  const uint32_t m = group_max_u32<16>(max_of_pair(magnitudes8(val)));
  s = act_to_f32(static_cast<uint16_t>(m), f16) / 448.0f;
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
  return make_uint2(w[0], w[1]);
}

// A workgroup of 256 serves the groups first_group ..., 16 at a time and NV times, read together: one group of a
// lane makes for waves so short that their starts (some three a nanosecond) are what a large batch waits for.
// From kFp8TwoGroups groups on two a lane: behind a launch that writes the rows, us, one / two / three / four: [24008, 2048] 24.7 /
// 23.6 / 23.4 / 24.4, [8192, 7168] 37.7 / 35.4 / 35.4 / 37.1, [2048, 2048] 6.7 / 6.8 / 6.7 / 6.9, [512, 768] 2.1 / 2.4 / 2.7 / 2.9; inside a
// layer of 3001 tokens the second quantisation 38.9 -> 31.3, the first, beside the routing, 21.2 -> 19.5.
constexpr long long kFp8TwoGroups = 1 << 16;
template <int NV>
__device__ __forceinline__ void quant_fp8_group128_body(const uint16_t* __restrict__ x, int64_t ld_x, int R, int C,
                                                        uint8_t* __restrict__ q, int64_t ld_q, float* __restrict__ scale,
                                                        uint32_t first_group, bool f16) {
  const uint32_t groups_per_row = C / 128, total = static_cast<uint32_t>(R) * groups_per_row;
  const int t = threadIdx.x & 15;
  Pack8 val[NV];
  uint32_t gid[NV], r[NV], g[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    gid[i] = first_group + i * 16 + (threadIdx.x >> 4);
    const uint32_t at = min(gid[i], total - 1);
    r[i] = at / groups_per_row;
    g[i] = at - r[i] * groups_per_row;
    val[i].v = *reinterpret_cast<const uint4*>(x + static_cast<size_t>(r[i]) * ld_x + g[i] * 128 + t * 8);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (gid[i] >= total) return;  // (a group's 16 lanes leave together)
    float s;
    *reinterpret_cast<uint2*>(q + static_cast<size_t>(r[i]) * ld_q + g[i] * 128 + t * 8) = quant8_fp8(val[i], f16, s);
    if (t == 0) scale[static_cast<size_t>(r[i]) * groups_per_row + g[i]] = s;
  }
}

}  // namespace kmoe
