// The GEMM launch for experts of several hundred rows (macro_tile.hip).
#pragma once
#include "kmoe_common.h"

namespace kmoe {

struct MacroParams {
  const int8_t* a;
  int64_t lda;           // bytes
  const float* a_max;    // int8: [a_rows] absmax
  const int32_t* row_src;
  uint32_t div_magic;    // ceil(2^32 / src_div) of the gather entries, 0 if they name rows themselves
  const int8_t* w;       // tiled
  const float* w_max;    // int8: [E, n] absmax
  const int32_t* lod;
  int32_t E, n, k;       // k in bytes
  uint16_t* y;
  int64_t ldy;
  const int8_t* w_tail;
  const float* w_max_tail;
  int32_t tail_row0, tail_rows, tail_src0;
  int32_t n_blocks;      // (the launcher's)
  int32_t m_major;       // order of an expert's items: as in tiled_gemm.hip
  int32_t low;           // fp8: tiles of 128 rows
  int32_t y_past;        // the results leave past the caches
  int32_t past;          // the weights of an expert with one tile are read past the caches (see buffer_stream_load16)
};
// Rows of K it takes: whole chunks of 128 bytes, twelve of its 64-byte steps at least (the first six store the tile before, the
// last six copy the next one's first steps). Experts, the tail among them: their row ranges lie in LDS beside the rings.
constexpr int kMacroTables = 3296, kMacroBlocks = 64;
inline bool macro_tile_takes(int kbytes, int E, bool tail) {
  return kbytes % 128 == 0 && kbytes >= 768 && 4 * (2 * E + 2 + (tail ? 1 : 0)) <= kMacroTables;
}
// Gather entries it divides by one multiplication: entry / div = high half of entry * magic, for every entry where the excess is at most 2.
inline bool macro_tile_divides(int div, uint32_t* magic) {
  *magic = div > 1 ? static_cast<uint32_t>(((1ull << 32) + div - 1) / div) : 0;
  return div <= 1 || static_cast<uint64_t>(*magic) * div - (1ull << 32) <= 2;
}
// kind 0: int8, 1: 16-bit, 2: fp8 block-scaled (a_max: [a_rows, k/128] scales, w_max: [E, n/128, k/128]; K of up to kMacroBlocks blocks;
// with SiLU-mul gate and up in whole blocks: n % 256 == 0). Arguments already checked as for the tile kernel.
int macro_tile(const MacroParams& p, int kind, bool swiglu, bool f16, int rows, hipStream_t s, int n_cu, const char* what);

}  // namespace kmoe
