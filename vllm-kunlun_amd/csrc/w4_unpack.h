// Packed 4-bit weights to 16-bit operands, in registers: shared by the weight-streaming kernel and the tile kernel.
//   value    bf16(float(c - 8) * scale), or with half activations half(c - 8) * scale in half arithmetic: the same bits
//            as unpacking first (kmoe_dequant_w4).
#pragma once
#include "kmoe_common.h"

namespace kmoe {

typedef int w4_v4i __attribute__((ext_vector_type(4)));
typedef _Float16 w4_v2h __attribute__((ext_vector_type(2)));

// What unpacking a lane's words needs of a group's scale.
// bf16: value (c - 8) s is ONE fused multiply-add on the code's bits read as a half. A nibble alone in the low 8 bits
// of a half is the subnormal c 2^-24 (in the upper half of a byte: c 2^-20), which v_fma_mix_f32 widens for free:
// c 2^-24 * s 2^24 - 8 s, whose product and sum are exact in f32 (a code has 4 significant bits, a scale 8), so the one
// rounding is the one to bf16. half: v_fma_mixlo_f16 would do the whole of it, but issues at half the rate (8.45 against
// 4.75 clocks per instruction and SIMD), so the code is OR-ed into the mantissa of 1024.0h (whose last place counts
// ones), 1032 subtracted exactly and one packed multiply rounds the product.
template <bool F16>
struct W4Scale;
template <>
struct W4Scale<false> {
  float lo, hi, m8;  // s 2^24, s 2^20, -8 s
  W4Scale() = default;
  __device__ explicit W4Scale(uint16_t bits) {
    const float s = bf16_to_f32(bits);
    lo = s * 0x1p24f;
    hi = s * 0x1p20f;
    m8 = s * -8.0f;
  }
};
template <>
struct W4Scale<true> {
  w4_v2h s2;
  W4Scale() = default;
  __device__ explicit W4Scale(uint16_t bits) {
    const _Float16 s = __builtin_bit_cast(_Float16, bits);
    s2 = w4_v2h{s, s};
  }
};

// 8 codes of one 4-byte word -> 8 bf16 values, value 2 j in the low half of register j. Five instructions put the nibbles
// into halves ((n0, n4), (n1, n5), (n2, n6), (n3, n7)), then one fused multiply-add per value and one rounding per pair:
// 17 where splitting the nibbles into bytes, building 128 + c from each byte, multiplying and rounding takes 23.
__device__ inline w4_v4i unpack8(uint32_t word, const W4Scale<false>& s) {
  const uint32_t up = word >> 8;
  const w4_v2h a = __builtin_bit_cast(w4_v2h, word & 0x000f000fu), b = __builtin_bit_cast(w4_v2h, word & 0x00f000f0u);
  const w4_v2h c = __builtin_bit_cast(w4_v2h, up & 0x000f000fu), d = __builtin_bit_cast(w4_v2h, up & 0x00f000f0u);
  w4_v4i out;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    out[2 * h] = static_cast<int>(pack2_bf16(__builtin_fmaf(static_cast<float>(a[h]), s.lo, s.m8),
                                             __builtin_fmaf(static_cast<float>(b[h]), s.hi, s.m8)));
    out[2 * h + 1] = static_cast<int>(pack2_bf16(__builtin_fmaf(static_cast<float>(c[h]), s.lo, s.m8),
                                                 __builtin_fmaf(static_cast<float>(d[h]), s.hi, s.m8)));
  }
  return out;
}

// The same 8 codes -> 8 half values: pair j is (code 2 j, code 2 j + 1) = byte j of lo and of hi.
template <int J>
__device__ inline int unpack2_half(uint32_t lo, uint32_t hi, w4_v2h s2) {
  // bytes, most significant first: zero, byte J of hi, zero, byte J of lo; then the exponent of 1024.0h on both
  const uint32_t bits =
      __builtin_amdgcn_perm(hi, lo, 0x0c000c00u | (static_cast<uint32_t>(4 + J) << 16) | static_cast<uint32_t>(J)) | 0x64006400u;
  const w4_v2h v = (__builtin_bit_cast(w4_v2h, bits) - (w4_v2h){(_Float16)1032.0f, (_Float16)1032.0f}) * s2;
  return __builtin_bit_cast(int, v);
}
__device__ inline w4_v4i unpack8(uint32_t word, const W4Scale<true>& s) {
  const uint32_t lo = word & 0x0f0f0f0fu;
  const uint32_t hi = (word >> 4) & 0x0f0f0f0fu;
  w4_v4i out;
  out[0] = unpack2_half<0>(lo, hi, s.s2);
  out[1] = unpack2_half<1>(lo, hi, s.s2);
  out[2] = unpack2_half<2>(lo, hi, s.s2);
  out[3] = unpack2_half<3>(lo, hi, s.s2);
  return out;
}

}  // namespace kmoe
