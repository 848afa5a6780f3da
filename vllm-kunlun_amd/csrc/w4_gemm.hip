// Grouped GEMM on 4-bit weights and bf16 activations (W4A16): the launch on tiles of 16 to 128 rows, and the choice
// between it and the weight-streaming kernel (stream_gemm.hip). In both the
// packed weights are unpacked in registers and fed to v_mfma_f32_16x16x32_bf16: a quarter of the
// bytes of the bf16 path; the unpacking (17 VALU instructions per 8 weights, 13 for half) is what bounds the
// streaming kernel once the bytes are that few, and what the tile kernel shares among its rows.
//
//   weights  [E][n][k/2] bytes, two codes per byte, low nibble first, code c means c - 8
//            (dequant_int4_native, quantization/kernels/quant_ops.py:71-86), re-arranged by
//            kmoe_tile_weights_i8(E, n, k/2): 1 KB blocks of 16 channels x 128 values. Lane
//            16 g + c of a wave reads 16 consecutive bytes of a block: the 32 values
//            k = 128 kb + 32 g + [0, 32) of channel c. Its t-th 4-byte word (8 values) is its
//            operand of the t-th MFMA of the block; the activation lane (g, row) supplies the
//            same 8 values of its row. So one MFMA step covers k = 32 g + 8 t + [0, 8) for
//            g = 0..3 - not a contiguous range, which the sum does not care about.
//   scales   [E][n][k/group] bf16; a group is a multiple of 32 values, so a lane needs ONE
//            scale per block: group (128 kb + 32 g) / group_size of its channel.
//   value    bf16(float(c - 8) * scale) (F16 instantiations: activations, scales and results are IEEE half, the
//            dtype dequant_int4_native itself produces; value = half(c - 8) * scale in half arithmetic): one
//            exact fused multiply-add and one rounding, the same bits as unpacking first (kmoe_dequant_w4).
#include <type_traits>
#include <utility>

#include "buffer_ops.h"
#include "kmoe_common.h"
#include "w4_unpack.h"

namespace kmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

struct W4Params {
  const uint16_t* a;  // [a_rows, k] bf16
  int64_t lda;
  const int32_t* row_src;
  int32_t src_div;
  const uint8_t* w;       // tiled packed codes
  const uint16_t* scale;  // [E, n, k / gs] bf16
  int32_t gs;
  int32_t gs_shift;       // log2(gs / 32) when gs / 32 is a power of two, else -1
  // Element strides inside the 16 x (k / gs) scales of a fragment (16 channels), which start at channel * (k / gs) in
  // both layouts. KMOE_S_ROWMAJOR: channel k / gs, group 1. KMOE_S_FRAG16 (kmoe_tile_scales_w4): channel 1, group 16 -
  // the scales a wave needs for one block are then 32 to 128 consecutive bytes: one cache line per load instruction
  // where the row-major layout touches 16 (one per channel), and consecutive LDS banks in the wave's copy.
  int32_t s_ch, s_g;
  const int32_t* lod;
  int32_t E, n, k;
  uint16_t* y;
  int64_t ldy;
};

constexpr int kWaves = 4;

// ---------------------------------------------------------------------------------------------------
// Tiles of 16, 32, 64, 96 or 128 rows. The unpacking of a weight word (17 VALU instructions per 8 values) is shared by
// the row fragments of the tile, one MFMA each; the kernel is bound by issuing both, at a quarter of the 16-bit weights'
// bytes. One workgroup: one tile of sorted rows of one expert x 4 waves x 4 fragments of 16 channels. Activations are
// copied global -> LDS asynchronously in 128-value blocks of K (256 bytes per row); every wave reads its A fragments
// from there. Weights go global -> registers, one or two blocks ahead; they never pass through LDS.

// Work item `item` = (m-tile, channel block) when every expert's rows are cut into tiles of kTileRows and the
// items are numbered m-tile by m-tile: expert, first row and channel block (false: no such item). The hardware
// deals workgroups to the 8 XCDs in turn, so workgroup b takes item (b % 8) * ceil(items / 8) + b / 8: the
// workgroups of one XCD, which share an L2, walk consecutive items - the channel blocks of one m-tile (the same
// activation rows) and the m-tiles of one expert (the same weights). Dealt the other way round, every activation
// row was fetched by six L2s (gate_up of the Qwen3 shape at 8192 tokens: 2.2 GB fetched for 0.5 GB of operands).
template <int kTileRows>
__device__ inline bool locate_w4_item(const W4Params& p, int n_blocks, int& e_out, int& row0_out, int& nb_out) {
  const int lane = lane_id();
  const int epl = (p.E + kWave - 1) / kWave;  // experts per lane
  const int e_begin = lane * epl;
  int local = 0;
  for (int i = 0; i < epl; ++i) {
    const int e = e_begin + i;
    if (e < p.E) local += (p.lod[e + 1] - p.lod[e] + kTileRows - 1) / kTileRows;
  }
  int incl = local;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  const int items = __shfl(incl, kWave - 1, kWave) * n_blocks;
  const int seg = (items + 7) >> 3;
  const int j = blockIdx.x >> 3;
  const int item = (blockIdx.x & 7) * seg + j;
  if (j >= seg || item >= items) return false;
  const int t = item / n_blocks;
  nb_out = item - t * n_blocks;
  int excl = incl - local;
  int found_e = -1, found_row = 0;
  if (t >= excl && t < incl) {
    for (int i = 0; i < epl; ++i) {
      const int e = e_begin + i;
      if (e >= p.E) break;
      const int lo = p.lod[e];
      const int tiles = (p.lod[e + 1] - lo + kTileRows - 1) / kTileRows;
      if (t < excl + tiles) {
        found_e = e;
        found_row = lo + (t - excl) * kTileRows;
        break;
      }
      excl += tiles;
    }
  }
  const int src_lane = __builtin_ctzll(__ballot(found_e >= 0));
  e_out = __shfl(found_e, src_lane, kWave);
  row0_out = __shfl(found_row, src_lane, kWave);
  return true;
}

// The four MFMAs of row fragment `mf`, left out if the tile has no rows there: a branch the compiler does not see, so the
// K loop stays one basic block (with a visible one the accumulators spill). The compare and the branch are the two
// wait states between the unpacking's last write and the first MFMA that reads it.
template <bool F16, int MF_INDEX>
__device__ __forceinline__ void mfma4_if_live(v4f (&c)[4], const v4i (&w)[4], const v4i& a, int live_frags) {
#define KMOE_W4_MFMA4(OP)                                                                                              \
  asm volatile("s_cmp_le_i32 %[live], %[mf]\n\t"                                                                       \
               "s_cbranch_scc1 1f\n\t" OP " %[c0], %[w0], %[a], %[c0]\n\t" OP " %[c1], %[w1], %[a], %[c1]\n\t" OP         \
               " %[c2], %[w2], %[a], %[c2]\n\t" OP " %[c3], %[w3], %[a], %[c3]\n"                                        \
               "1:"                                                                                                    \
               : [c0] "+v"(c[0]), [c1] "+v"(c[1]), [c2] "+v"(c[2]), [c3] "+v"(c[3])                                     \
               : [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]), [a] "v"(a), [live] "s"(live_frags),     \
                 [mf] "n"(MF_INDEX)                                                                                    \
               : "scc")
  if constexpr (F16)
    KMOE_W4_MFMA4("v_mfma_f32_16x16x32_f16");
  else
    KMOE_W4_MFMA4("v_mfma_f32_16x16x32_bf16");
#undef KMOE_W4_MFMA4
}

template <class F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(f, std::make_integer_sequence<int, N>{});
}

// MF: 16-row fragments of a tile (1, 2, 4, 6, 8). The short tiles keep one block of weights and activations ahead and
// run three or four workgroups per CU instead of more blocks and two: the unpacking of one wave then has three others'
// waits and MFMAs to run beside. Layer, Kimi-K2 dims with groups of 32: 2048 tokens on 64-row tiles 2650 us with four
// blocks and two workgroups, 2450 with two and three; 700 tokens on 32-row tiles 1786, where 16-row passes of the
// streaming kernel took 2776 and 64-row tiles with two workgroups 2101; 128 tokens on 16-row tiles 1537 (streaming 1599).
// The tall tiles' accumulators leave room for two.
constexpr int w4_workgroups(int MF) { return MF <= 2 ? 4 : (MF == 4 ? 3 : 2); }
// R: blocks of weights (registers) and of activations (LDS) in the rings. A stage waits for its own block, passes a
// barrier, requests block kb + R - 1 of both and multiplies. The waits count the loads of weights and activations, so blocks past the end
// are requested as well, out of the descriptors' range: they fetch nothing. The scales' chunks are copied under a uniform branch; no wait counts
// on them, and one that still counts them waits for more than it has to, never for less.
constexpr int w4_ring(int MF) { return MF == 6 ? 3 : 2; }
// PAST: the weights are read past the caches (see buffer_stream_load16), where nearly every expert has one m-tile: always at 16 and 32
// rows, at 64 rows up to 50 rows per expert. Layer, us, ordinary / past the caches: Qwen3 dims 128 tokens 78.8 / 75.9, cold 84.0 / 79.8,
// Kimi-K2 dims 64 tokens 1232 / 1191, 2048 2418 / 2390; with several tiles per expert their siblings miss: Qwen3 dims 2048 tokens 238 / 247.
// (A hot expert's tiles do, too: Kimi-K2 dims, +2.0 on the logits of 8 experts, 1000 tokens 2120 / 2135, 2000 2639 / 2666, but 400 1799 / 1779. A
// choice per tile between two loops, as the tile kernel of the other formats has, took 2627 at 2000, but more elsewhere: 400 even 1623 -> 1677,
// Qwen3 dims, 400 with hot experts 111 -> 119.)
// CHUNKED: the scales come CB blocks at a time, by asynchronous copies into LDS of the wave's own, one chunk ahead, and from there to
// registers one block ahead (a group of 32: 512 consecutive bytes of each fragment). Asked for block by block and lane by lane they were a third
// of the load instructions for a ninth of the bytes, in pieces of 128: with nothing but its loads the gate_up launch of Kimi-K2 dims, 2048 tokens, took
// 1275 us with them and 1160 without. For layouts KMOE_S_FRAG16 with groups of a power of two; others keep those loads. With rows past a tile's
// end no longer fetched and a step unpacked right before its MFMAs (ten registers less, the other waves' MFMAs run beside it), layer, us,
// before / after: Kimi-K2 dims 64 tokens 1167 / 1124, 150 1517 / 1466, 400 1662 / 1608, 800 1807 / 1768, 2048 2416 / 2374; Qwen3 dims 64 75.4 / 74.1,
// 240 88.3 / 85.5, 400 101.0 / 98.5, 1000 145.7 / 145.4, 4096 403 / 400.
constexpr int w4_chunk(int MF) { return MF >= 6 ? 2 : 4; }
template <int MF, bool SWIGLU, bool F16, bool PAST, bool CHUNKED>
__global__ __launch_bounds__(kWaves* kWave, w4_workgroups(MF)) void w4_tile_kernel(const W4Params p) {
  constexpr int NF = 4, R = w4_ring(MF), CB = w4_chunk(MF);
  constexpr int kScaleBytes = NF * CB * 128;  // a chunk of groups of 32; fewer bytes of larger groups
  constexpr int kTileRows = 16 * MF;
  constexpr int NFH = SWIGLU ? NF / 2 : NF;
  constexpr int NA = kTileRows / 4 / kWaves;  // asynchronous copies per wave and block: 4 rows (1 KB) each
  constexpr int kWaveRows = 4 * NA;           // tile rows a wave copies
  constexpr int kBufBytes = kTileRows * 256;
  // Row r of a block sits at r * 256; its 16-byte vector v at position v ^ swizzle(r % 16): the rows of a fragment read
  // fall on different bank groups without padding, which the asynchronous copies (1 KB of consecutive LDS bytes per
  // instruction) could not write. A read serves lanes 0-3, 12-15 and 20-27 together, then 4-11, 16-19 and 28-31, and
  // so on: rows 0-3 and 12-15 of one vector with rows 4-11 of the vector four further. The swizzle has to keep those
  // apart: it sends the first eight rows to 0-7 and the others to 8-15 (r itself makes every pair of them collide:
  // four clocks more per read).
  auto swizzle = [](int r) { return r ^ ((r & 4) << 1); };
  __shared__ __attribute__((aligned(1024))) int8_t lds_a[R][kBufBytes];
  __shared__ __attribute__((aligned(1024))) int8_t lds_s[CHUNKED ? kWaves : 1][2][CHUNKED ? kScaleBytes : 16];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int n_half = SWIGLU ? p.n / 2 : p.n;
  int e, row0, nb;
  if (!locate_w4_item<kTileRows>(p, (n_half + kWaves * NFH * 16 - 1) / (kWaves * NFH * 16), e, row0, nb)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  nb = __builtin_amdgcn_readfirstlane(nb);
  const int row_end = min(p.lod[e + 1], row0 + kTileRows);
  const int live_frags = __builtin_amdgcn_readfirstlane((row_end - row0 + 15) / 16);  // row fragments that hold rows
  const int col_base = (nb * kWaves + wave) * NFH * 16;
  const int kblocks = p.k / 128;
  const int groups = p.k / p.gs;
  constexpr uint32_t kRange = 0xfffffff0u;
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, kRange, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.w + static_cast<size_t>(e) * p.n * (p.k / 2)), 0, kRange, 0x00020000);
  const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.scale + static_cast<size_t>(e) * p.n * groups), 0,
                                                                          CHUNKED ? static_cast<uint32_t>(p.n * groups) * 2u : kRange, 0x00020000);

  uint32_t woff[NF], soff[NF];  // scalar: the fragment's first block; vector: the lane's channel in the fragment's scales
  bool wok[NF];
  int col[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int fh = SWIGLU ? f % NFH : f;
    const int c = col_base + fh * 16;
    wok[f] = c < n_half;
    col[f] = (SWIGLU && f >= NFH) ? n_half + c : c;
    const int ch0 = wok[f] ? col[f] : 0;  // fragments past the last channel read fragment 0: never stored
    woff[f] = static_cast<uint32_t>(ch0 / 16) * kblocks * 1024u;
    soff[f] = static_cast<uint32_t>(ch0) * groups * 2u;
  }
  // copy i of this wave fills tile rows kWaveRows wave + 4 i + lane / 16; the lane fetches the vector that belongs at its position
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int tr = kWaveRows * wave + 4 * i + lg;
    const int r = row0 + tr;
    const int rr = r < row_end ? r : row0;
    const int src = p.row_src ? p.row_src[rr] / p.src_div : rr;
    // < 4 GiB: host-checked; rows past the end are not read (and never stored)
    aoff[i] = r < row_end ? static_cast<uint32_t>(src) * static_cast<uint32_t>(p.lda * 2) + ((li ^ swizzle(tr & 15)) << 4) : kRange;
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)&lds_a[0][0]));
  // fragment reads of MFMA step t: row li (+ 16 per fragment: same row % 16), vector 4 lg + t
  uint32_t fa[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) fa[t] = lds_base + li * 256 + (((4 * lg + t) ^ swizzle(li)) << 4);
  v4f acc[MF][NF];
#pragma unroll
  for (int mf = 0; mf < MF; ++mf)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[mf][f] = (v4f){0.f, 0.f, 0.f, 0.f};
  v4i wbuf[R][NF];
  int sbuf[CHUNKED ? 1 : R][NF];  // (the upper halves are not looked at)
  const uint32_t lane16 = lane * 16u;
  const uint32_t lane_s = li * p.s_ch * 2u;
  // chunked scales: a fragment's groups of a chunk are s_frag consecutive bytes; copy j of a chunk takes bytes 1024 j + 16 lane of the
  // wave's fragments, one behind the other
  constexpr int NS = CHUNKED ? kScaleBytes / 1024 : 1;
  const int s_frag = 32 * max(1, (4 * CB) >> max(p.gs_shift, 0));
  uint32_t s_off[NS];
  const uint32_t s_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)&lds_s[CHUNKED ? wave : 0][0][0]));
  if constexpr (CHUNKED) {
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int at = j * 1024 + lane * 16, f = at / s_frag;
      uint32_t off = kRange;
#pragma unroll
      for (int g = 0; g < NF; ++g) off = f == g ? soff[g] + static_cast<uint32_t>(at & (s_frag - 1)) : off;
      s_off[j] = off;
    }
  }
  auto first_group = [&](int kb) __attribute__((always_inline)) { return (4 * (kb & ~(CB - 1))) >> p.gs_shift; };  // of the chunk of block kb
  // the chunk that begins with block kb, which has to exist: the descriptor ends with the expert's scales, and a scalar offset beyond its
  // end would wrap in the range check (limit minus offset); what a last chunk has beyond it is not fetched
  auto dma_s = [&](int kb) __attribute__((always_inline)) {
    const uint32_t at = static_cast<uint32_t>(first_group(kb)) * 32u;
#pragma unroll
    for (int j = 0; j < NS; ++j) buffer_load16_to_lds(s_rsrc, (lds_ptr_t)&lds_s[CHUNKED ? wave : 0][kb / CB & 1][j * 1024], s_off[j], at);
  };
  // the scales of block kb, which the caller has seen land in LDS; usable behind the wait for a younger LDS read and hold_s(), which keeps their
  // registers theirs until then, also where nothing uses the values (the last block asks for the next one's, too)
  auto request_s = [&](int kb) __attribute__((always_inline)) {
    const uint32_t at = s_lds + static_cast<uint32_t>((kb / CB & 1) * kScaleBytes + (((4 * kb + lg) >> p.gs_shift) - first_group(kb)) * 32 + li * 2);
#pragma unroll
    for (int f = 0; f < NF; ++f) asm volatile("ds_read_u16 %0, %1" : "=v"(sbuf[0][f]) : "v"(at + static_cast<uint32_t>(f * s_frag)) : "memory");
  };
  auto hold_s = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < NF; ++f) asm volatile("" : "+v"(sbuf[0][f])::"memory");
  };
  auto load_w = [&](int slot, int kb) __attribute__((always_inline)) {
    const bool live = kb < kblocks;
    uint32_t s_at = 0;
    if constexpr (!CHUNKED) {
      const int g32 = 4 * kb + lg;  // this lane's 32 values of the block
      s_at = lane_s + static_cast<uint32_t>((p.gs_shift >= 0 ? g32 >> p.gs_shift : g32 / (p.gs / 32)) * p.s_g) * 2u;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const uint32_t at = live ? woff[f] + static_cast<uint32_t>(kb) * 1024u : kRange;
      wbuf[slot][f] = PAST ? buffer_stream_load16(w_rsrc, lane16, at) : buffer_load16(w_rsrc, lane16, at);
      if constexpr (!CHUNKED) sbuf[slot][f] = __builtin_amdgcn_raw_buffer_load_b16(s_rsrc, s_at, live ? soff[f] : kRange, 0);
    }
  };
  auto dma_a = [&](int buf, int kb) __attribute__((always_inline)) {
    const uint32_t at = kb < kblocks ? static_cast<uint32_t>(kb) * 256u : kRange;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      buffer_load16_to_lds(a_rsrc, (lds_ptr_t)&lds_a[buf][(kWaveRows * wave + 4 * i) * 256], aoff[i], at);
  };
  // One block: word t of a lane's 16 packed bytes is its operand of MFMA step t; the activation lane (lg, row)
  // supplies values 32 lg + 8 t + [0, 8) of the block, i.e. vector 4 lg + t of the row's 16.
  auto compute = [&](int kb, auto slot_tag) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_tag)::value, ss = CHUNKED ? 0 : slot;
    const W4Scale<F16> sc[NF] = {W4Scale<F16>(sbuf[ss][0]), W4Scale<F16>(sbuf[ss][1]), W4Scale<F16>(sbuf[ss][2]), W4Scale<F16>(sbuf[ss][3])};
    if constexpr (CHUNKED) {
      __builtin_amdgcn_sched_barrier(0);
      request_s(kb + 1);
    }
    // Row fragments are read two ahead, across the steps: fragment i = t MF + mf of the block's 4 MF.
    v4i af[3];
    auto request = [&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value;
      // (the offset field of an LDS read reaches 64 KB)
      constexpr int off = slot * kBufBytes + (i % MF) * 16 * 256;
      af[i % 3] = off < 65536 ? lds_read16_raw<(off < 65536 ? off : 0)>(fa[i / MF])
                              : lds_read16_raw<(off < 65536 ? 0 : off - 65536)>(fa[i / MF] + 65536u);
    };
    request(std::integral_constant<int, 0>{});
    request(std::integral_constant<int, 1>{});
    v4i wv[NF];
    __builtin_amdgcn_sched_barrier(0);
    static_for<4 * MF>([&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value;
      constexpr int t = i / MF, mf = i % MF;
      if constexpr (i + 2 < 4 * MF) {
        request(std::integral_constant<int, i + 2>{});
        lds_wait<2>(af[i % 3]);
      } else if constexpr (i + 1 < 4 * MF) {
        lds_wait<1>(af[i % 3]);
      } else {
        lds_wait<0>(af[i % 3]);
      }
      if constexpr (mf == 0) {
#pragma unroll
        for (int f = 0; f < NF; ++f) wv[f] = unpack8(static_cast<uint32_t>(wbuf[slot][f][t]), sc[f]);
      }
      mfma4_if_live<F16, mf>(acc[mf], wv, af[i % 3], live_frags);
      __builtin_amdgcn_sched_barrier(0);  // (all the unpacking of a block at once would not fit the registers)
    });
    if constexpr (CHUNKED) hold_s();
  };
  auto stage = [&](int kb, auto u_tag) __attribute__((always_inline)) {
    constexpr int u = decltype(u_tag)::value;
    vmem_wait<(R - 2) * (NA + (CHUNKED ? 1 : 2) * NF)>();  // the loads of a wave younger than those the stage needs
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (CHUNKED) {
      if ((kb & (CB - 1)) == 0 && kb + CB < kblocks) dma_s(kb + CB);  // (the waits do not count on these copies)
    }
    dma_a((u + R - 1) % R, kb + R - 1);
    load_w((u + R - 1) % R, kb + R - 1);
    __builtin_amdgcn_sched_barrier(0);
    compute(kb, u_tag);
  };
  if constexpr (CHUNKED) dma_s(0);
#pragma unroll
  for (int i = 0; i < R - 1; ++i) {
    dma_a(i, i);
    load_w(i, i);
  }
  if constexpr (CHUNKED) {  // (the first stage waits for the loads behind these anyway)
    vmem_wait<0>();
    request_s(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    hold_s();
  }
  // (no exit inside the body: with one the accumulators do not fit the registers)
  int kb = 0;
  for (; kb + R <= kblocks; kb += R)
    static_for<R>([&](auto u) __attribute__((always_inline)) { stage(kb + decltype(u)::value, u); });
  static_for<R - 1>([&](auto u) __attribute__((always_inline)) {
    if (kb + decltype(u)::value < kblocks) stage(kb + decltype(u)::value, u);
  });

  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMAs' results, which the compiler does not know to wait for
  __builtin_amdgcn_sched_barrier(0);
  // epilogue: as the streaming kernel - round to the activation type, optional SiLU-mul on the rounded values
  auto pack2 = [](float lo, float hi) { return F16 ? pack2_half(lo, hi) : pack2_bf16(lo, hi); };
  auto low = [](uint32_t v) { return act_to_f32(static_cast<uint16_t>(v), F16); };
  auto high = [](uint32_t v) { return act_to_f32(static_cast<uint16_t>(v >> 16), F16); };
#pragma unroll
  for (int mf = 0; mf < MF; ++mf) {
    if (mf >= live_frags) continue;  // (wave-uniform)
    const int r = row0 + mf * 16 + li;
#pragma unroll
    for (int f = 0; f < NFH; ++f) {
      const int c0 = col[f] + lg * 4;
      const v4f g = acc[mf][f];
      uint2 out = make_uint2(pack2(g[0], g[1]), pack2(g[2], g[3]));
      if constexpr (SWIGLU) {
        const v4f u = acc[mf][f + NFH];
        const uint32_t u0 = pack2(u[0], u[1]), u1 = pack2(u[2], u[3]);
        out.x = pack2(silu_hw(low(out.x)) * low(u0), silu_hw(high(out.x)) * high(u0));
        out.y = pack2(silu_hw(low(out.y)) * low(u1), silu_hw(high(out.y)) * high(u1));
      }
      if (wok[f] && r < row_end) *reinterpret_cast<uint2*>(p.y + static_cast<size_t>(r) * p.ldy + c0) = out;
    }
  }
}

template <int MF, bool SWIGLU, bool PAST = (MF <= 2)>
int launch_w4_tile(const W4Params& p, int rows, bool f16, hipStream_t s) {
  constexpr int kTileRows = 16 * MF;
  constexpr int NFH = SWIGLU ? 2 : 4;
  const int n_half = SWIGLU ? p.n / 2 : p.n;
  // an upper bound of the work items (m-tiles x channel blocks), a multiple of 8
  const int n_blocks = ceil_div(n_half, kWaves * NFH * 16);
  const int items = (rows / kTileRows + min(p.E, rows)) * n_blocks;
  const dim3 grid(ceil_div(items, 8) * 8);
  const bool chunked = p.gs_shift >= 0 && p.s_g == 16 && reinterpret_cast<uintptr_t>(p.scale) % 16 == 0 &&
                       static_cast<int64_t>(p.n) * (p.k / p.gs) < (1ll << 30);
  if (tracing_kernels())
    note_kernel("w4_tile_kernel<%d-row tiles, %s, %s, %d per CU, scales by %s>", kTileRows, SWIGLU ? "SiLU-mul" : "plain",
                f16 ? "f16" : "bf16", w4_workgroups(MF), chunked ? "chunks" : "lanes");
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kWaves * kWave), 0, s, p); };
  if (f16) chunked ? launch(w4_tile_kernel<MF, SWIGLU, true, PAST, true>) : launch(w4_tile_kernel<MF, SWIGLU, true, PAST, false>);
  else chunked ? launch(w4_tile_kernel<MF, SWIGLU, false, PAST, true>) : launch(w4_tile_kernel<MF, SWIGLU, false, PAST, false>);
  return check_launch("kmoe_grouped_gemm_w4a16");
}

// scales [rows = E * n][groups] -> per 16 rows [groups][16]
__global__ __launch_bounds__(256) void tile_scales_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                         long long total, int groups) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;  // index into dst
  if (i >= total) return;
  const long long frag = i / (16LL * groups);
  const int r = static_cast<int>(i - frag * 16LL * groups);
  const int g = r >> 4, c = r & 15;
  dst[i] = src[(frag * 16 + c) * groups + g];
}

}  // namespace

// Layers as [hidden x intermediate], time on 16-row tiles (whose launch needs the sort's, and which read a scale once per chunk of the contraction) over time on 16-row passes of
// the streaming kernel (which sorts the pairs on the way and splits the contraction over its waves): even load / +2.0 on the logits of eight
// experts / every token on the same experts.
// Rows beyond 4096 values. Up to 16 tokens no expert needs a second pass, and tiles lack workgroups where tokens share experts: 160 experts of
// [5120 x 1536], top 6, 8 tokens 1.09 / 1.08 / 1.58, 64 of [6144 x 3072], top 4, 10 1.03 / 1.10 / 1.59, 32 of [8192 x 2048], top 4, 6 1.19 / 1.14 /
// 1.92, Kimi-K2 dims 10 1.06 / 1.02 / 1.36, 16 0.97 / 1.03 / 1.08. From 17 on: Kimi-K2 dims 20 0.95 / 0.97 / 0.86, 32 0.96 / 0.92 / 0.68, 160 of [5120 x
// 1536] 24 0.98 / 0.88 / 1.00, 160 of [6144 x 2560], top 8, 20 0.96 / 0.97 / 0.77.
// Shorter rows, where the sort's launch counts: only from 49 tokens on, when an expert that most of them choose takes four passes. Qwen3 dims 20
// 1.08 / 1.01 / 0.84, 40 1.01 / 0.97 / 0.69, 49 to 64 1.00 / 0.90 to 0.82 / 0.64 to 0.53; 128 of [3072 x 1024], top 8, 36 1.03 / 0.99 / -, 56 0.99 / 0.92 /
// 0.61; 64 of [3584 x 2560], top 6, 40 1.05 / 0.97 / 0.75.
// Few workgroups, even load: 32 of [2048 x 1024], top 4, (256) 20 to 32 tokens 1.09, 16 of [8192 x 4096], top 2, (512) 8 1.18, 12 1.08, 32 of [7168 x
// 2048], top 8, 5 tokens (350) 1.10, 8 (450) 1.04.
bool w4_gate_up_streams(int rows, int rows_hint, long long tokens, int E, int n, int k) {
  const int expected = expected_rows(rows, rows_hint);
  const int avg = ceil_div(expected, E);
  const bool fills = static_cast<long long>(min(expected, E)) * ceil_div(n / 2, kWaves * 32) > 512;  // two workgroups a CU
  if (k > 4096) return avg <= 1 && !(tokens > 16 && expected > E / 4 && fills);
  return avg <= 4 && !(tokens > 48 && avg > 2 && fills);
}

}  // namespace kmoe

using namespace kmoe;

extern "C" int kmoe_tile_scales_w4(const uint16_t* src, uint16_t* dst, int E, int n, int groups, kmoe_stream_t stream) {
  KMOE_REQUIRE(src && dst && src != dst, KMOE_ERR_NULL, "tile_scales_w4: NULL pointer, or in place");
  KMOE_REQUIRE(E >= 1 && n >= 16 && n % 16 == 0 && groups >= 1, KMOE_ERR_SHAPE, "tile_scales_w4: E=%d n=%d groups=%d", E, n, groups);
  const long long total = static_cast<long long>(E) * n * groups;
  hipLaunchKernelGGL(tile_scales_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, as_stream(stream), src,
                     dst, total, groups);
  return check_launch("kmoe_tile_scales_w4");
}

extern "C" int kmoe_grouped_gemm_w4a16(const kmoe_gemm_w4_args* a, kmoe_stream_t stream) {
  return grouped_gemm_w4a16_checked(a, stream, nullptr, nullptr, a && !a->row_src ? a->rows : -1);
}

int kmoe::grouped_gemm_w4a16_checked(const kmoe_gemm_w4_args* a, kmoe_stream_t stream, const StreamScan* scan,
                                     const StreamSlots* slots, long long a_rows) {
  KMOE_REQUIRE(a, KMOE_ERR_NULL, "grouped_gemm_w4a16: NULL args");
  KMOE_REQUIRE(a->a && a->w && a->w_scale && (a->lod || scan) && a->y, KMOE_ERR_NULL, "grouped_gemm_w4a16: NULL pointer");
  KMOE_REQUIRE(a->E >= 1 && a->rows >= 0, KMOE_ERR_SHAPE, "grouped_gemm_w4a16: E=%d rows=%d", a->E, a->rows);
  const bool swiglu = a->act == KMOE_ACT_SWIGLU;
  KMOE_REQUIRE(a->act == KMOE_ACT_NONE || swiglu, KMOE_ERR_UNSUPPORTED, "grouped_gemm_w4a16: act=%d", a->act);
  KMOE_REQUIRE(a->w_layout == KMOE_W_TILED, KMOE_ERR_UNSUPPORTED,
               "grouped_gemm_w4a16: the packed weights must be tiled (kmoe_tile_weights_i8 on [E, n, k/2] bytes)");
  KMOE_REQUIRE(a->k >= 128 && a->k % 128 == 0 && a->n >= 16 && a->n % (swiglu ? 32 : 16) == 0, KMOE_ERR_SHAPE,
               "grouped_gemm_w4a16: n=%d k=%d (need k %% 128 == 0, n %% %d == 0)", a->n, a->k, swiglu ? 32 : 16);
  KMOE_REQUIRE(a->group_size >= 32 && a->group_size % 32 == 0 && a->k % a->group_size == 0, KMOE_ERR_SHAPE,
               "grouped_gemm_w4a16: group_size=%d must be a multiple of 32 that divides k=%d", a->group_size, a->k);
  KMOE_REQUIRE(a->lda >= a->k && a->lda % 8 == 0 && reinterpret_cast<uintptr_t>(a->a) % 16 == 0, KMOE_ERR_SHAPE,
               "grouped_gemm_w4a16: activations need 16-byte aligned rows (lda=%lld)", static_cast<long long>(a->lda));
  KMOE_REQUIRE(a->ldy % 4 == 0 && a->ldy >= (swiglu ? a->n / 2 : a->n), KMOE_ERR_SHAPE, "grouped_gemm_w4a16: ldy=%lld",
               static_cast<long long>(a->ldy));
  KMOE_REQUIRE(!a->row_src || a->src_div >= 1, KMOE_ERR_SHAPE, "grouped_gemm_w4a16: src_div=%d", a->src_div);
  KMOE_REQUIRE(reinterpret_cast<uintptr_t>(a->w_scale) % 4 == 0, KMOE_ERR_SHAPE, "grouped_gemm_w4a16: misaligned scales");
  KMOE_REQUIRE(a->act_dtype == KMOE_DT_BF16 || a->act_dtype == KMOE_DT_F16, KMOE_ERR_UNSUPPORTED,
               "grouped_gemm_w4a16: act_dtype=%d unknown", a->act_dtype);
  const bool f16 = a->act_dtype == KMOE_DT_F16;
  if (a->rows == 0 && !scan) return KMOE_OK;
  const int q = a->group_size / 32;
  int shift = -1;
  if ((q & (q - 1)) == 0)
    for (shift = 0; (1 << shift) < q; ++shift) {}
  KMOE_REQUIRE(a->scale_layout == KMOE_S_ROWMAJOR || a->scale_layout == KMOE_S_FRAG16, KMOE_ERR_UNSUPPORTED,
               "grouped_gemm_w4a16: scale_layout=%d unknown", a->scale_layout);
  const int groups = a->k / a->group_size;
  const bool frag16 = a->scale_layout == KMOE_S_FRAG16;
  const W4Params p{a->a, a->lda, a->row_src, a->src_div, a->w, a->w_scale, a->group_size, shift,
                   frag16 ? 1 : groups, frag16 ? 16 : 1, a->lod, a->E, a->n, a->k, a->y, a->ldy};
  hipStream_t s = as_stream(stream);
  int mf = a->variant;
  // the tile kernel reaches a source row (gathered or not: below `rows`) through a 32-bit byte offset, the streaming
  // kernel's split launches too (gathered rows of a caller may lie anywhere: those take its other launches)
  const bool tile_ok = w4_rows_fit_32(a->rows, a->lda, a->k);
  const bool stream_fits_32 = a_rows >= 0 && w4_rows_fit_32(a_rows, a->lda, a->k);
  if (mf == 0) {
    // The streaming kernel where it sorts the pairs itself or has a column of workgroups per pair, or for a gate_up of
    // few rows; its plain down launch is 4 to 7 % behind 16-row tiles from one row per expert on (Qwen3 dims, 16 / 32 /
    // 64 tokens: 19.7 / 24.2 / 26.7 us against 18.8 / 23.7 / 24.9). Tiles by the rows an expert gets under uniform routing, with
    // headroom for the spread - an expert with more rows unpacks its weights again, one with fewer leaves its tile's
    // accumulators unused and workgroups out of the CU. Layer, us, 16- / 32- / 64-row tiles, Qwen3 dims: 112 tokens (7 rows)
    // 80.0 / 81.7 / 88.2, 144 (9) 87.2 / 82.5 / 89.8, 330 (21) 119 / 95.8 / 100, 360 (23) 123 / 105 / 101; Kimi-K2 dims:
    // 350 (8) 1688 / 1703 / 1840, 1000 (21) 2681 / 2002 / 2064, 1200 (25) 2987 / 2155 / 2137. 64- / 96- / 128-row, Qwen3
    // dims: 768 (48) 140.7 / 141.0 / 149.1, 832 (52) 146.2 / 144.5 / 152.0, 1152 (72) 183 / 168 / 170, 1300 (82) 192 / 189 /
    // 176, 1800 (113) 225 / 251 / 224, 2048 (128) 252 / 263 / 262, 2300 (144) 275 / 270 / 290, 2560 (160) 291 / 285 / 305,
    // 3072 (192) 333 / 335 / 324, 8192 (512) 776 / 756 / 716.
    const int avg = ceil_div(expected_rows(a->rows, a->rows_hint), a->E);
    const long long tokens = a_rows >= 0 ? a_rows : ceil_div(a->rows, a->src_div);
    if (scan || slots || (swiglu && w4_gate_up_streams(a->rows, a->rows_hint, tokens, a->E, a->n, a->k))) mf = 1;
    else if (!tile_ok) mf = avg <= 13 ? 1 : (avg <= 20 ? 2 : 4);
    else if (avg <= 22) mf = avg <= 8 ? 16 : 32;
    else if (avg <= 112) mf = avg <= 50 ? 64 : (avg <= 76 ? 96 : 128);
    else mf = avg <= 136 ? 64 : (avg <= 176 ? 96 : 128);
  }
  if (mf == 8) mf = 128;
  const bool tile = mf == 16 || mf == 32 || mf == 64 || mf == 96 || mf == 128;
  KMOE_REQUIRE((!scan && !slots) || mf == 1, KMOE_ERR_UNSUPPORTED, "grouped_gemm_w4a16: only the weight-streaming kernel sorts the pairs itself");
  if (tile)
    KMOE_REQUIRE(tile_ok, KMOE_ERR_SHAPE, "grouped_gemm_w4a16: the tile kernel addresses the activations with 32 bits (rows=%d lda=%lld)",
                 a->rows, static_cast<long long>(a->lda));
  switch (mf) {
    case 1:
    case 2:
    case 4: return stream_gemm_w4(a, s, mf, scan, slots, stream_fits_32);
    case 16: return swiglu ? launch_w4_tile<1, true>(p, a->rows, f16, s) : launch_w4_tile<1, false>(p, a->rows, f16, s);
    case 32: return swiglu ? launch_w4_tile<2, true>(p, a->rows, f16, s) : launch_w4_tile<2, false>(p, a->rows, f16, s);
    case 64:
      if (ceil_div(expected_rows(a->rows, a->rows_hint), a->E) <= 50)
        return swiglu ? launch_w4_tile<4, true, true>(p, a->rows, f16, s) : launch_w4_tile<4, false, true>(p, a->rows, f16, s);
      return swiglu ? launch_w4_tile<4, true>(p, a->rows, f16, s) : launch_w4_tile<4, false>(p, a->rows, f16, s);
    case 96: return swiglu ? launch_w4_tile<6, true>(p, a->rows, f16, s) : launch_w4_tile<6, false>(p, a->rows, f16, s);
    case 128: return swiglu ? launch_w4_tile<8, true>(p, a->rows, f16, s) : launch_w4_tile<8, false>(p, a->rows, f16, s);
    default:
      return fail(KMOE_ERR_UNSUPPORTED, "grouped_gemm_w4a16: variant=%d must be 0, 1, 2, 4, 8, 16, 32, 64, 96 or 128", a->variant);
  }
}
