// The operand formats of the decode kernels.
#pragma once
#include "kmoe_common.h"

namespace kmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

enum class Fmt { I8, F8, BF16, F16, W4, W4H };  // W4H: half activations, scales and results
constexpr const char* fmt_name(Fmt f) {
  constexpr const char* names[] = {"i8", "fp8", "bf16", "f16", "4-bit", "4-bit, f16"};
  return names[static_cast<int>(f)];
}

}  // namespace
}  // namespace kmoe
