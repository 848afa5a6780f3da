// How the launches of a few tokens keep rows in LDS (no GPU code).
#pragma once

namespace kmoe {

// Bytes from one row of `values` values to the next: the values, where they have any (fp8) the scales of their groups of 128, and 16
// bytes more, so that rows start in other banks. Lanes read 16 bytes at a time: every row starts on a multiple of them, also
// where the scales do not fill one (fp8 rows of 768 values have 24 bytes of them).
constexpr int few_row_pitch(int values, int value_bytes, bool group_scales) {
  return (values * value_bytes + (group_scales ? values / 128 * 4 : 0) + 15) / 16 * 16 + 16;
}

}  // namespace kmoe
