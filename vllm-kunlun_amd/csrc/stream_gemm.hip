// Weight-streaming grouped GEMM for the decode regime (a handful of rows per expert), on int8 (W8A8), fp8-e4m3
// (128x128 / 1x128 block scales), bf16, half and packed 4-bit weights: HBM-bound, every weight byte is read once, MFMA is
// ~5% busy.
//
// A wave needs no LDS, no barrier and no address arithmetic beyond a stride in its main loop:
//   weights  "tiled": [E][n/16][k bytes/64] blocks of 1 KB; inside a block byte
//            256*g + 16*c + t is channel c (of 16), byte 16*g + t of the block's 64 bytes of K (g = 0..3) —
//            i.e. exactly what lane 16*g + c feeds the MFMA. A wave reads 1 KB
//            of consecutive bytes per block and the next block follows
//            directly: one long sequential stream per 16 output channels. int8, bf16 and half: a block is an MFMA
//            step; fp8: a step is two blocks, one 128-value scale block, whose partial sums are scaled and added in f32;
//            4-bit: a step is one block of 128 values: a lane's 16 bytes are values 32 g + [0, 32) of its channel, its
//            t-th word unpacked (w4_unpack.h) its operand of the t-th of four MFMAs, one group scale for all of them.
//   activations: lane (g, r) reads the same bytes of K of its row r. int8: "chunk-major" [k/64][rows][64 B], one
//            chunk per step: the rows of an expert are consecutive (down GEMM: 1 KB of consecutive bytes per step) or a
//            gather of 64-byte pieces (gate_up GEMM: one half cache line per row and
//            step; with 16-byte chunks a gathered load touched four times as many
//            lines, which cost the DeepSeek-V3 gate_up launch 9 %). The other formats: row-major, 64 to 256
//            consecutive bytes of a row per step.
// Each wave owns NF channel fragments and keeps D MFMA steps of loads in flight.
#include <type_traits>

#include "buffer_ops.h"
#include "formats.h"
#include "kmoe_common.h"
#include "pair_scan.h"
#include "quant_body.h"
#include "w4_unpack.h"

namespace kmoe {
namespace {

struct StreamParams {
  const int8_t* a;
  int64_t a_row, a_step;  // bytes between rows; between the MFMA steps of a row
  int32_t a_rows;         // chunk-major activations: their rows
  const float* a_aux;     // I8: row maxes; F8: [row][k/128] scales
  const int32_t* row_src;
  int32_t src_div;
  const int8_t* w;        // tiled
  const float* w_aux;     // I8: [E][n] maxes; F8: [E][n/128][k/128] scales
  const int32_t* lod;
  int32_t E, n, kbytes;
  uint16_t* y;
  int64_t ldy;
  int32_t* acc_out;
  const int8_t* w_tail;
  const float* w_aux_tail;
  int32_t tail_row0, tail_rows, tail_src0;
  int32_t f16;  // outputs (and the rounding of gate and up before SiLU-mul) in IEEE half instead of bf16
  int32_t rotate;  // every wave starts its K range at a step of its own (see stream_gemm_i8)
  StreamScan scan;    // SCAN instantiations: the routed pairs' expert ids instead of lod / row_src
  StreamQuant quant;  // QUANT instantiations: the rows as bf16 / half values instead of codes and row maxes
  // W4: group scales. Element strides inside the 16 x (k / group) scales of a fragment (16 channels), which start at
  // channel * (k / group) in both layouts. KMOE_S_ROWMAJOR: channel k / group, group 1. KMOE_S_FRAG16
  // (kmoe_tile_scales_w4): channel 1, group 16 - what a step needs is then 32 to 128 consecutive bytes: one cache line
  // per load instruction where the row-major layout touches 16 (one per channel).
  const uint16_t* w_scale;
  int32_t groups, s_ch, s_g;
  int32_t gs32, gs_shift;  // values per group / 32, and its log2 if it is a power of two, else -1
  StreamSlots slots;  // n > 0: a column of workgroups per pair instead of per expert (pair_scan.h)
  int32_t late_w;  // the first weight steps are requested when the column's rows are known
};

constexpr int kWaves = 4;
constexpr int kQuantStride = kStreamQuantMaxK + 16;  // bytes between the rows of the LDS copy: row li starts 16 li B into the banks

// KS: the workgroup's 4 waves split K KS ways (KS = 1, 2, 4): 4/KS waves own
// different channels, KS waves share channels and add their partial
// sums through LDS in a fixed order (int8: exact). More, shorter streams: a finer-grained tail on small layers.
//
// SCAN: the launch does the stable sort by expert itself. Every workgroup reads all the routed pairs' expert ids
// (p.scan.ids, a few KB from L2, a quarter per wave, kScanBatch loads in flight), counts the ids below its expert
// (its first sorted row) and lists the pairs that chose it, in order (its rows): what lod and row_src would have
// told it, after one memory round trip instead of two dependent ones and without the sort's launch before this one.
// The workgroups of channel block 0 also write the sort's outputs (lod, expert_m, moe_index, sorted_src) for the
// launches that follow.
//
// QUANT: the launch quantises its rows itself (the int8 down projection of a decode-sized layer with k <= 1024). Per
// 16-row pass the workgroup's four waves read the pass's live rows as bf16 / half values (p.quant.act), one row
// per wave at a time, and leave absmax and codes - the arithmetic of quant_i8_rows_body, hence its bits - in LDS,
// where the K loop reads its row fragments; a and a_aux are not read. The workgroups of channel block 0 also write
// codes (chunk-major) and row maxes where the quantiser's launch would have left them. Built for four waves per
// SIMD (see stream_gemm_i8).
template <Fmt FMT, int MF, int NF, bool SWIGLU, int D, int KS, bool SCAN = false, bool QUANT = false>
__global__ __launch_bounds__(kWaves* kWave, QUANT ? 4 : 1) void stream_gemm_kernel(const StreamParams p) {
  static_assert(!SCAN || kWaves == kScanWaves, "scan_pairs is written for four waves");
  static_assert(!QUANT || (FMT == Fmt::I8 && MF == 1 && KS == 1 && !SWIGLU && !SCAN), "QUANT: the 16-row int8 down-projection shape only");
  using acc_t = typename std::conditional<FMT == Fmt::I8, v4i, v4f>::type;
  constexpr bool W4 = FMT == Fmt::W4 || FMT == Fmt::W4H;
  constexpr bool kRows32 = W4 && KS > 1;  // activation rows through 32-bit offsets (stream_gemm_w4 sees to it that they fit)
  constexpr int V = FMT == Fmt::F8 ? 2 : 1;  // 1 KB blocks of weights per step
  constexpr int AV = W4 ? 4 : V;             // 16-byte vectors of activations per lane and step ...
  constexpr int kAVStride = W4 ? 16 : 64, kALane = W4 ? 64 : 16;  // ... bytes between them, between the lane groups
  constexpr int NFH = SWIGLU ? NF / 2 : NF;
  constexpr int TM = 16 * MF;
  constexpr int WN = kWaves / KS;  // waves along the channel dimension
  __shared__ acc_t red[KS > 1 ? (KS - 1) * WN * MF * NF * kWave : 1];
  __shared__ typename std::conditional<SCAN, PairScanLds, int>::type scan_lds;
  __shared__ __attribute__((aligned(16))) int8_t qrows[QUANT ? 16 * kQuantStride : 16];
  __shared__ float qmax[16];
  const int lane = lane_id();
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_id / KS;   // channel group of this wave
  const int wk = wave_id % KS;     // K part of this wave
  const int li = lane & 15;
  const int lg = lane >> 4;
  const bool f16 = FMT == Fmt::F16 || FMT == Fmt::W4H || ((FMT == Fmt::I8 || FMT == Fmt::F8) && p.f16 != 0);

  // Columns: one per expert (or, with slots, one per pair and - in the launch that sorts - one that writes lod), all of
  // the expert's rows; beyond: one 16*MF-row slice of the tail expert each.
  const int column = blockIdx.y;
  const int n_cols = p.slots.n > 0 ? p.slots.n + (SCAN ? 1 : 0) : p.E;
  const bool tail = column >= n_cols;
  int e = tail ? p.E : column;
  if (p.slots.n > 0 && !tail) {
    if constexpr (SCAN) {
      if (column == p.slots.n) {
        if (blockIdx.x == 0) publish_lod(p.scan, p.E, scan_lds);
        return;
      }
    }
    e = p.slots.ids[column];
  }
  const int8_t* w_base = tail ? p.w_tail : p.w + static_cast<size_t>(e) * p.n * p.kbytes;
  const size_t n_aux = FMT == Fmt::F8 ? static_cast<size_t>(p.n / 128) * (p.kbytes / 128) : p.n;
  const float* w_aux = tail ? p.w_aux_tail : p.w_aux + static_cast<size_t>(e) * n_aux;

  const int n_half = SWIGLU ? p.n / 2 : p.n;
  const int ksteps = p.kbytes / (64 * V);
  const int col_base = (blockIdx.x * WN + wave) * NFH * 16;
  // whole wave has nothing to do (no barriers when KS == 1; with QUANT it stays for the quantisation and its barriers)
  const bool idle = KS == 1 && col_base >= n_half;
  if (idle && !QUANT && !SCAN) return;
  const int kb_begin = (ksteps * wk) / KS;
  const int kb_end = (ksteps * (wk + 1)) / KS;
  // With p.rotate a wave walks its K range from a start step of its own, wrapping round: int32 sums do not depend
  // on the order, and waves that were dispatched together no longer read addresses that differ by a
  // multiple of the fragment stride.
  const int klen = kb_end - kb_begin;
  const unsigned wave_key = (static_cast<unsigned>(blockIdx.y) * gridDim.x + blockIdx.x) * kWaves + wave_id;
  const int rot = FMT == Fmt::I8 && p.rotate && klen > 1
                      ? static_cast<int>(((wave_key * 2654435761u) >> 12) % static_cast<unsigned>(klen)) : 0;
  auto kb_of = [&](int i) {
    const int s = i + rot;
    return kb_begin + (s >= klen ? s - klen : s);
  };

  // The weight loads of the K loop are raw buffer loads, a lane offset that stays and a scalar offset per step: no address
  // arithmetic on the vector unit and 20 to 40 registers less than with pointers, and no select after a load, which
  // would wait for it (with pointers the two kinds of load in load_w_step took twice the time of one). 4-bit weights: the
  // activations too where their offsets fit 32 bits (kRows32), rows past the end lying past the descriptor's end: they
  // read zero and fetch nothing (Kimi-K2 dimensions, 128 tokens: layer 1674 -> 1577 us, Qwen3 93 -> 90).
  __amdgpu_buffer_rsrc_t wr[NF];
  bool wok[NF];
  int col[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int fh = SWIGLU ? f % NFH : f;
    const int c = col_base + fh * 16;
    wok[f] = c < n_half;
    col[f] = (SWIGLU && f >= NFH) ? n_half + c : c;
    const size_t frag = wok[f] ? col[f] / 16 : 0;
    const int frag_bytes = ksteps * (V * 1024);
    wr[f] = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(w_base + frag * frag_bytes), 0, wok[f] ? frag_bytes : 0, 0x00020000);
  }

  // The first weight steps are requested before anything else: their addresses depend on the block's coordinates
  // only, while the rows do on two dependent loads (the expert's row range, then the gather indices). All
  // workgroups of a launch do the same work, so they start and end in rounds, and a round that begins with those
  // loads leaves the memory queue idle for their latency. Done where a wave's K range is short (a workgroup lives
  // a few microseconds: Qwen3 decode down projection 42.8 -> 40.4 us); with long ranges it changes nothing for the
  // better (DeepSeek-V3 decode: +0.4 %), so those keep the plain order. So do 16-bit launches
  // with a column per expert and fewer than three rows per expert (p.late_w): a third of an expert's bytes is much to ask
  // for where it may have no rows (Qwen3 dims, layer: 16 tokens 150 -> 143 us, with +2.0 on the logits of 8 experts 115
  // -> 104; 48 tokens 204.5 / 205.6); the columns of pairs rarely have none (6 tokens 79 / 81).
  const bool w_first = QUANT || W4 || (klen * V < 16 && !p.late_w);
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.a), 0, 0xfffffff0, 0x00020000);
  v4i wreg[D][NF][V];
  v4i areg[D][MF][AV];
  float asc[D][MF];  // F8: the rows' scales of the step
  uint16_t gsc[D][NF];  // W4: the channels' group scales of the step
  const uint16_t* sp[NF];
  if constexpr (W4) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      sp[f] = p.w_scale + (static_cast<size_t>(e) * p.n + (wok[f] ? col[f] : 0)) * p.groups + li * p.s_ch;
  }
  // The weights are read past the caches (see buffer_stream_load16), unless the workgroup will read them again: an expert's
  // rows beyond TM take another pass. Qwen3 dims, int8, +2.0 on the logits of 8 experts, layer with ordinary loads / past the
  // caches always / past them on an expert's last pass: 64 tokens 127 / 130 / 115 us, 140 tokens 182 / 203 / 163. Nor where another
  // workgroup reads them: the slices of a tail expert. DeepSeek-V3 dims, layer with all slices past the caches / none: int8 23 tokens
  // 838.7 / 831.7 us, 64 1462 / 1449, 128 1652 / 1630; fp8 23 843.9 / 835.2, 128 1663 / 1647, 250 1812 / 1781; 8 tokens (one slice) level.
  // (A single layer called again and again, of which the 256 MB memory-side cache holds what a batch hits, is faster with ordinary loads,
  // among other layers it is not. Qwen3 dims, layer with ordinary loads / past the caches, called again at once; cold: 4-bit 8 tokens
  // 41.9 / 43.7; 48.4 / 47.0, 16 55.6 / 61.2; 66.7 / 64.6, int8 8 49.1 / 50.9; 58.6 / 57.5.)
  const bool slices = tail && p.tail_rows > TM;
  bool once = !slices;
  auto load_w_step = [&](int slot, int kb) {
    auto load = [&](auto past) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const uint32_t at = static_cast<uint32_t>(kb) * (V * 1024) + v * 1024;
          wreg[slot][f][v] = past ? buffer_stream_load16(wr[f], lane * 16, at) : buffer_load16(wr[f], lane * 16, at);
        }
    };
    if (once) load(std::true_type{});
    else load(std::false_type{});
    if constexpr (W4) {
      const int g32 = 4 * kb + lg;  // this lane's 32 values of the step
      const int g = p.gs_shift >= 0 ? g32 >> p.gs_shift : g32 / p.gs32;
#pragma unroll
      for (int f = 0; f < NF; ++f) gsc[slot][f] = sp[f][g * p.s_g];
    }
  };
  if (w_first) {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < klen) load_w_step(d, kb_of(d));
  }
  // F8: lane l holds the block scale of step kb_begin + l for each fragment (the host keeps klen <= 64)
  float wsc[NF];
  if constexpr (FMT == Fmt::F8) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      wsc[f] = wok[f] ? w_aux[static_cast<size_t>(col[f] / 128) * ksteps + min(kb_begin + lane, ksteps - 1)] : 0.0f;
  }
  __builtin_amdgcn_sched_barrier(0);

  int row_begin, row_end;
  ListedRows listed = {};  // SCAN: the expert's rows
  if (tail) {
    row_begin = p.tail_row0 + (column - n_cols) * TM;
    row_end = min(p.tail_row0 + p.tail_rows, row_begin + TM);
  } else if constexpr (SCAN) {
    listed = scan_pairs(p.scan, e, p.E, scan_lds, blockIdx.x == 0);
    row_begin = listed.begin;
    row_end = listed.end;
    if (p.slots.n > 0) {
      if (listed.pair(scan_lds, 0) != column) row_end = row_begin;  // an earlier pair's column serves this expert
      if (blockIdx.x == 0 && threadIdx.x == 0) p.scan.slot_rows[column] = make_int2(row_begin, row_end);
    }
    if (idle) return;  // (KS == 1: no barrier after the scan's)
  } else if (p.slots.n > 0) {
    const int2 range = p.slots.rows[column];
    row_begin = range.x;
    row_end = range.y;
  } else {
    row_begin = p.lod[e];
    row_end = p.lod[e + 1];
  }
  if (SCAN && idle) return;  // (a tail slice's waves without channels; the routed ones left after the barrier)
  if (row_begin >= row_end) return;  // (an expert without rows has asked for a few KB of its weights in vain)

  for (int row0 = row_begin; row0 < row_end; row0 += TM) {
    if (QUANT) {
      if (row0 != row_begin) __syncthreads();  // the pass before has read its fragments
      const int nvec = p.kbytes / 8;  // vectors of 8 values per row: at most 2 per lane
      // (both loads of a row go out together, lanes past its end reading its last vector again; with the loads under conditions
      // of their own, one after the other, and the general arithmetic 128 tokens of the Qwen3 dims took 113.3 us, now 110.9)
#pragma unroll 1
      for (int q = 0; q < 4; ++q) {
        const int qi = wave_id + 4 * q;
        const int r = row0 + qi;
        if (r >= row_end) break;  // wave-uniform
        const uint4* src = reinterpret_cast<const uint4*>(p.quant.act + static_cast<size_t>(r) * p.quant.ld);
        Pack8 val[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) val[i].v = src[min(lane + i * kWave, nvec - 1)];
        RowScale rs = row_scale_i8(group_max_u32<kWave>(max_of_pair(max_magnitudes(magnitudes8(val[0]), magnitudes8(val[1])))), f16);
        if (!rs.numbers) {
          rs.amax = group_max<kWave>(fmaxf(amax8(val[0], f16), amax8(val[1], f16)));
          rs.inv = rs.amax > 0.0f ? 127.0f / rs.amax : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int v = lane + i * kWave;
          if (v < nvec) {
            const uint2 w = quant8_i8_of(val[i], rs, f16);
            *reinterpret_cast<uint2*>(&qrows[qi * kQuantStride + v * 8]) = w;
            if (blockIdx.x == 0)
              *reinterpret_cast<uint2*>(p.quant.codes + (static_cast<size_t>(v >> 3) * p.a_rows + r) * 64 + (v & 7) * 8) = w;
          }
        }
        if (lane == 0) {
          qmax[qi] = rs.amax;
          if (blockIdx.x == 0) p.quant.amax[r] = rs.amax;
        }
      }
      __syncthreads();
      if (idle) continue;
    }
    uint32_t aoff[MF];
    const int8_t* ap[MF];
    const float* asp[MF];
    int srow[MF];
#pragma unroll
    for (int mf = 0; mf < MF; ++mf) {
      const int r = row0 + mf * 16 + li;
      if constexpr (SCAN)
        srow[mf] = r < row_end ? (tail ? p.tail_src0 + r - p.tail_row0 : listed.pair(scan_lds, r - row_begin) / p.src_div) : -1;
      else
        srow[mf] = r < row_end ? (tail ? p.tail_src0 + r - p.tail_row0 : (p.row_src ? p.row_src[r] / p.src_div : r)) : -1;
      const size_t at = srow[mf] >= 0 ? srow[mf] : 0;
      // rows past the end read row 0 (valid memory, results never stored) or nothing
      ap[mf] = p.a + at * p.a_row + lg * kALane;
      if constexpr (kRows32)
        aoff[mf] = srow[mf] >= 0 ? static_cast<uint32_t>(srow[mf]) * static_cast<uint32_t>(p.a_row) + lg * kALane : 0xfffffff0u;
      if constexpr (FMT == Fmt::F8) asp[mf] = p.a_aux + at * ksteps;
    }
    acc_t acc[MF][NF];
#pragma unroll
    for (int mf = 0; mf < MF; ++mf)
#pragma unroll
      for (int f = 0; f < NF; ++f) acc[mf][f] = acc_t{0, 0, 0, 0};

    auto load_a_step = [&](int slot, int kb) {
      if (QUANT) return;  // (read from LDS where it is used)
#pragma unroll
      for (int mf = 0; mf < MF; ++mf) {
#pragma unroll
        for (int v = 0; v < AV; ++v) {
          if constexpr (kRows32)
            areg[slot][mf][v] = buffer_load16(ar, aoff[mf], static_cast<uint32_t>(kb) * static_cast<uint32_t>(p.a_step) + v * kAVStride);
          else
            areg[slot][mf][v] = *reinterpret_cast<const v4i*>(ap[mf] + kb * p.a_step + v * kAVStride);
        }
        if constexpr (FMT == Fmt::F8) asc[slot][mf] = asp[mf][kb];
      }
    };
    once = !slices && __builtin_amdgcn_readfirstlane(row_end - row0) <= TM;
    auto load_step = [&](int slot, int kb) {
      load_w_step(slot, kb);
      load_a_step(slot, kb);
    };

#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < klen) {
        if (row0 != row_begin || !w_first) load_w_step(d, kb_of(d));  // (the first pass may have them already)
        load_a_step(d, kb_of(d));
      }

    // I8, 16-row tiles: the scales are asked for before the K loop. In the epilogue each load waited for the one before it,
    // behind the weights of the launch's other workgroups: Qwen3 dims, layer, 16 tokens 82.0 -> 80.2 us, 64 102.1 -> 101.2.
    // (Taller tiles have no registers to spare.)
    constexpr bool kEarly = FMT == Fmt::I8 && MF == 1;
    float a_max = 0.0f;
    float4 w_max[NF];
    if constexpr (kEarly) {
      if constexpr (!QUANT) a_max = p.a_aux[max(srow[0], 0)];
#pragma unroll
      for (int f = 0; f < NF; ++f) w_max[f] = *reinterpret_cast<const float4*>(w_aux + (wok[f] ? col[f] : 0) + lg * 4);
    }

    for (int i0 = 0; i0 < klen; i0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int kb = i0 + d;
        if (kb < klen) {
          if constexpr (FMT == Fmt::F8) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              const float sw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wsc[f]), kb));
              const v8i wv = __builtin_shufflevector(wreg[d][f][0], wreg[d][f][V - 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
              for (int mf = 0; mf < MF; ++mf) {
                const v8i av = __builtin_shufflevector(areg[d][mf][0], areg[d][mf][V - 1], 0, 1, 2, 3, 4, 5, 6, 7);
                const v4f blk = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv, av, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0,
                                                                               0x7f7f7f7f, 0, 0x7f7f7f7f);
                const float s = asc[d][mf] * sw;
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[mf][f][q] = __builtin_fmaf(blk[q], s, acc[mf][f][q]);
              }
            }
          } else if constexpr (W4) {
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              const W4Scale<FMT == Fmt::W4H> s(gsc[d][f]);
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const v4i wv = unpack8(static_cast<uint32_t>(wreg[d][f][0][t]), s);
#pragma unroll
                for (int mf = 0; mf < MF; ++mf) {
                  if constexpr (FMT == Fmt::W4)
                    acc[mf][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wv),
                                                                         __builtin_bit_cast(v8bf, areg[d][mf][t]), acc[mf][f], 0, 0, 0);
                  else
                    acc[mf][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wv),
                                                                        __builtin_bit_cast(v8h, areg[d][mf][t]), acc[mf][f], 0, 0, 0);
                }
              }
            }
          } else {
#pragma unroll
            for (int mf = 0; mf < MF; ++mf)
#pragma unroll
              for (int f = 0; f < NF; ++f) {
                if constexpr (FMT == Fmt::I8)
                  acc[mf][f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                      wreg[d][f][0],
                      QUANT ? *reinterpret_cast<const v4i*>(&qrows[li * kQuantStride + kb_of(kb) * 64 + lg * 16]) : areg[d][mf][0],
                      acc[mf][f], 0, 0, 0);
                else if constexpr (FMT == Fmt::BF16)
                  acc[mf][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wreg[d][f][0]),
                                                                       __builtin_bit_cast(v8bf, areg[d][mf][0]), acc[mf][f], 0, 0, 0);
                else
                  acc[mf][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wreg[d][f][0]),
                                                                      __builtin_bit_cast(v8h, areg[d][mf][0]), acc[mf][f], 0, 0, 0);
              }
          }
          if (kb + D < klen) load_step(d, kb_of(kb + D));
          // F8, K split two ways (long streams, many columns): a step's loads stay ahead of the next step's wait and scaling, where the
          // compiler would sink them (DeepSeek-V3 dims, layer, 8 tokens 393 -> 389 us, 23 898 -> 891, 64 1469 -> 1462; other formats level). Not where K
          // is whole or split four ways: 64 experts of [2816 x 2048], top 6, layer, 32 tokens 93.5 -> 98.4 us with it in the split launches, 100.3 in
          // all; 100 of [1024 x 1024], top 8, 44.6 -> 48.3; 16 of [8192 x 4096], top 2, 138.1 -> 136.6; level with four channel fragments a wave.
          if constexpr (FMT == Fmt::F8 && KS == 2) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }

    if (KS > 1) {  // add the K parts: waves wk > 0 park their sums in LDS, wave wk == 0 collects
      if (wk > 0) {
#pragma unroll
        for (int mf = 0; mf < MF; ++mf)
#pragma unroll
          for (int f = 0; f < NF; ++f)
            red[(((wk - 1) * WN + wave) * MF * NF + mf * NF + f) * kWave + lane] = acc[mf][f];
      }
      __syncthreads();
      if (wk == 0) {
#pragma unroll
        for (int part = 1; part < KS; ++part)
#pragma unroll
          for (int mf = 0; mf < MF; ++mf)
#pragma unroll
            for (int f = 0; f < NF; ++f)
              acc[mf][f] += red[(((part - 1) * WN + wave) * MF * NF + mf * NF + f) * kWave + lane];
      }
      if (row0 + TM < row_end) __syncthreads();  // red is reused by the next m-tile
      if (wk > 0) continue;
    }

#pragma unroll
    for (int mf = 0; mf < MF; ++mf) {
      const int r = row0 + mf * 16 + li;
      if (r >= row_end) continue;
      float sa = 1.0f;
      if constexpr (FMT == Fmt::I8) sa = (QUANT ? qmax[li] : kEarly ? a_max : p.a_aux[srow[mf]]) / 127.0f;
#pragma unroll
      for (int f = 0; f < NFH; ++f) {
        if (!wok[f]) continue;
        const int c0 = col[f] + lg * 4;
        uint16_t yv[4];
        auto finish = [&](const acc_t& a, int ff, uint16_t(&out)[4]) {
          if constexpr (FMT == Fmt::I8) {
            const int cc = col[ff] + lg * 4;
            const float4 wm = kEarly ? w_max[ff] : *reinterpret_cast<const float4*>(w_aux + cc);
            const float sw[4] = {wm.x / 127.0f, wm.y / 127.0f, wm.z / 127.0f, wm.w / 127.0f};
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q] = f32_to_act((static_cast<float>(a[q]) * sa) * sw[q], f16);
            if (p.acc_out) *reinterpret_cast<v4i*>(p.acc_out + static_cast<size_t>(r) * p.n + cc) = a;
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q] = f32_to_act(a[q], f16);
          }
        };
        finish(acc[mf][f], f, yv);
        if constexpr (SWIGLU) {
          uint16_t uv[4];
          finish(acc[mf][f + NFH], f + NFH, uv);
#pragma unroll
          for (int q = 0; q < 4; ++q) yv[q] = f32_to_act(silu_hw(act_to_f32(yv[q], f16)) * act_to_f32(uv[q], f16), f16);
        }
        const uint2 packed = make_uint2(yv[0] | (static_cast<uint32_t>(yv[1]) << 16),
                                        yv[2] | (static_cast<uint32_t>(yv[3]) << 16));
        *reinterpret_cast<uint2*>(p.y + static_cast<size_t>(r) * p.ldy + c0) = packed;
      }
    }
  }
}

template <Fmt FMT, int MF, int NF, bool SWIGLU, int D, int KS = 1, bool SCAN = false, bool QUANT = false>
int launch_stream(const StreamParams& p, hipStream_t s) {
  constexpr int NFH = SWIGLU ? NF / 2 : NF;
  const int n_half = SWIGLU ? p.n / 2 : p.n;
  const int cols = p.slots.n > 0 ? p.slots.n + (SCAN ? 1 : 0) : p.E;
  const dim3 grid(ceil_div(n_half, (kWaves / KS) * NFH * 16), cols + (p.w_tail ? ceil_div(p.tail_rows, 16 * MF) : 0));
  if (tracing_kernels())
    note_kernel("stream_gemm_kernel<%s, %d rows per pass, %d channel fragments per wave, %s, %d steps in flight, K split %d%s%s%s%s>",
                fmt_name(FMT), 16 * MF, NF, SWIGLU ? "SiLU-mul" : "plain", D, KS, SCAN ? ", sorts the pairs itself" : "",
                QUANT ? ", quantises its rows itself" : "", p.slots.n > 0 ? ", a column per pair" : "",
                (FMT == Fmt::W4 || FMT == Fmt::W4H) && KS > 1 ? ", 32-bit row offsets" : "");
  hipLaunchKernelGGL((stream_gemm_kernel<FMT, MF, NF, SWIGLU, D, KS, SCAN, QUANT>), grid, dim3(kWaves * kWave), 0, s, p);
  return check_launch("kmoe_grouped_gemm (stream)");
}

// The shapes of a 16-row launch, from its dimensions alone (`blocks`: workgroups of four waves side by side):
// K is split across the waves of a workgroup when its streams are long enough to share: more, shorter streams balance
// the tail (measured: +6..12% at k = 2048). Batches of a few tokens take the same shapes: with a column of workgroups per
// pair (Qwen3, one token: layer 53 -> 24 us, its launches no longer mostly workgroups of experts without rows) keeping
// a wave's whole K range in flight (8 steps) gains nothing at one token and loses 10 to 25 % from four tokens on.
// Figures below are the layer's time over its time without the branch, even load / +2.0 on the logits of eight experts / every token on the same
// experts (samples of one prompt), layers as [hidden x intermediate].
// (1) 16-bit gate_up launches with a column per expert keep four steps in flight, whose weights are twice the bytes and nothing to work on: Qwen3 dims
// 16 tokens 0.99 / 0.98 / 0.99, 64 0.99 / 0.97 / 0.95, 160 0.99 / 0.95 / 0.92, 32 of [7168 x 2048], top 8, 8 0.99 / 0.98 / 0.91, of [2048 x 1024], top 4, 24
// 0.98 / 0.92 / 1.03. Not with a column per
// pair (Qwen3 dims 8 tokens 1.00 / 0.99 / 1.03; 128 of [1024 x 768], top 8, 8 1.02 / 1.08 / 1.16), nor on rows whose first steps are asked for before the
// workgroup knows its rows (w_first; 64 of [1024 x 512], top 8, 24 0.99 / 0.99 / 1.10), nor on rows of 4096 and 8192 values and beyond (16 of [4096 x
// 4096], top 2, 32 1.03 / 0.99 / 1.02, of [8192 x 8192] 1.03), nor in launches of fewer workgroups than CUs (a rank's 16 of the 128 experts of Qwen3 dims, 32
// 1.04 / 1.01 / 1.00).
// (2) 16-bit columns of fewer than 64 pairs in a layer too large for the first rule, long rows: K split four ways at full depth. 160 of [5120 x 1536],
// top 6, 3 tokens 0.95 / 0.94 / 0.95, 10 0.98 / 0.96 / 0.91, 64 of [4096 x 2048], top 8, 5 0.96 / 0.93 / 0.94, 64 of [6144 x 3072], top 4, 8 0.97 / 0.97 / 0.89,
// 128 of [3072 x 4096], top 8, 4 0.98 / 0.99 / 0.97, 6 0.98 / 0.98 / 1.03. More columns read shared weights too often ([3072 x 4096], 12 tokens 0.99 / 0.99 /
// 1.16), and so do shorter rows (128 of [2048 x 3072], top 8, gate_up so too, 6 0.99 / 0.97 / 1.06; [5120 x 1536], down launch so too, 8 0.99 / 1.02 / 1.28). int8
// and fp8 gain 0 to 2 % and lose up to 24 where tokens share experts: DeepSeek-V3 dims int8 5 tokens 0.99 / 0.99 / 0.97, 16 1.00 / 1.00 / 1.05, 128 of
// [4096 x 4096], top 4, 8 1.00 / 0.98 / 1.12, 16 1.00 / 0.99 / 1.24, fp8 16 1.00 / 1.00 / 1.18.
// (3) From four rows per expert on every workgroup of a large gate_up launch reads rows enough for them to count: waves of four channel fragments, K
// split four ways, halve the workgroups that read them, where rows are long (int8 beyond 4096 codes, fp8 beyond 6144 and below 8192). Even load / hot
// experts: DeepSeek-V3 dims int8 128 tokens (4 rows) 1.00 / 1.00, 160 0.99 / 1.00, 250 0.97 / 0.98, 320 0.96 / 0.97, fp8 128 1.00 / 0.99, 250 0.98 / 0.98;
// 160 of [5120 x 1536], top 6, int8 112 1.00 / 0.95, 250 0.98 / 0.95; 128 of [7168 x 2048], top 8, int8 64 1.00 / 0.98, 160 0.97 / 0.96, fp8 96 1.00 / 0.96;
// 128 of [5120 x 5120], top 6, int8 160 0.99 / 1.01. Split two ways an expert's further passes weigh more: DeepSeek-V3 dims int8 250 0.97 / 1.01, 128 of
// [7168 x 2048] 96 0.99 / 1.02. Shorter rows, two ways: 64 of [4096 x 2048], top 8, int8 56 1.00 / 1.02, 128 of [3072 x 4096], top 8, 112 1.00 / 1.02, 256 of
// [2048 x 2048], top 8, 144 1.01 / 1.04, 128 of [4096 x 4096], top 4, 200 0.98 / 1.02. fp8 rows of 8192 values: 16 of [8192 x 8192], top 2, 40 1.08 / 1.09, 64 of [8192 x
// 3072], top 4, 80 1.06 / 1.01. (The fp8 fence, below, changes nothing here: 0.998 to 1.002.)
template <Fmt FMT, bool SWIGLU, bool SCAN>
int launch_rows16(const StreamParams& p, int rows, hipStream_t s) {
  constexpr int V = FMT == Fmt::F8 ? 2 : 1;
  const int ksteps = p.kbytes / 64;
  const int n_half = SWIGLU ? p.n / 2 : p.n;
  const int blocks = p.E * ceil_div(n_half, kWaves * (SWIGLU ? 1 : 2) * 16);
  constexpr bool k16 = FMT == Fmt::BF16 || FMT == Fmt::F16;
  if constexpr (k16 && SWIGLU) {  // (1)
    if (p.slots.n == 0 && ksteps >= 64 && ksteps < 256 && ksteps != 128 && blocks >= 256 && blocks < 2048) return launch_stream<FMT, 1, 2, SWIGLU, 4, 4, SCAN>(p, s);
  }
  if (ksteps >= 24 && blocks < 2048) return launch_stream<FMT, 1, 2, SWIGLU, 2, 4, SCAN>(p, s);
  if constexpr (k16 && SWIGLU == SCAN) {  // (2): a gate_up launch with columns of pairs sorts them, a down launch never does
    if (p.slots.n > 0 && p.slots.n < 64 && ksteps >= (SWIGLU ? 96 : 64)) return launch_stream<FMT, 1, 2, SWIGLU, 4, 4, SCAN>(p, s);
  }
  if constexpr (SWIGLU && (FMT == Fmt::I8 || FMT == Fmt::F8)) {  // (3)
    if ((FMT == Fmt::I8 ? ksteps > 64 : ksteps > 96 && ksteps < 128) && rows >= 4ll * p.E) return launch_stream<FMT, 1, 4, SWIGLU, 4 / V, 4, SCAN>(p, s);
  }
  if (ksteps >= 24) return launch_stream<FMT, 1, 2, SWIGLU, 4 / V, 2, SCAN>(p, s);
  return launch_stream<FMT, 1, 2, SWIGLU, 4 / V, 1, SCAN>(p, s);
}

// [E][n][k] row-major -> tiled blocks; one thread moves 16 bytes.
__global__ void tile_weights_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst, int n, int k,
                                    long long total_vec) {
  const long long v = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (v >= total_vec) return;
  const int ksteps = k / 64;
  const int lane = static_cast<int>(v & 63);
  const long long blk = v >> 6;  // (e * n/16 + nb) * ksteps + kb
  const int kb = static_cast<int>(blk % ksteps);
  const long long frag = blk / ksteps;  // e * n/16 + nb
  const long long row = frag * 16 + (lane & 15);
  const int kk = kb * 64 + (lane >> 4) * 16;
  *reinterpret_cast<uint4*>(dst + v * 16) = *reinterpret_cast<const uint4*>(src + row * k + kk);
}

int check_scan(const StreamScan* scan, bool swiglu, int variant, const int32_t* row_src, int rows) {
  KMOE_REQUIRE(swiglu && variant == 0 && row_src == nullptr && scan->ids && scan->lod && scan->expert_m &&
                   scan->moe_index && scan->sorted_src && scan->n_pairs == rows && rows <= kStreamScanMaxPairs,
               KMOE_ERR_UNSUPPORTED, "grouped_gemm (stream): not a launch that can sort the pairs itself");
  KMOE_REQUIRE(!scan->slot_rows || rows <= kStreamSlotMaxPairs, KMOE_ERR_UNSUPPORTED,
               "grouped_gemm (stream): %d pairs are too many for a column each", rows);
  return KMOE_OK;
}

StreamSlots slots_of(const StreamScan* scan, const StreamSlots* slots) {
  if (scan) return scan->slot_rows ? StreamSlots{scan->ids, scan->slot_rows, scan->n_pairs} : StreamSlots{};
  return slots ? *slots : StreamSlots{};
}

}  // namespace

int stream_gemm_i8(const kmoe_gemm_i8_args* a, hipStream_t s, const StreamScan* scan, const StreamQuant* quant,
                   const StreamSlots* slots) {
  StreamParams p{a->a, 64, static_cast<int64_t>(a->a_rows) * 64, a->a_rows, a->a_max, a->row_src, a->src_div, a->w, a->w_max,
                 a->lod, a->E,     a->n,     a->k,       a->y,       a->ldy, a->acc_out,
                 a->w_tail, a->w_max_tail, a->tail_row0, a->tail_rows, a->tail_src0, a->act_dtype == KMOE_DT_F16,
                 // A fragment's blocks are k / 64 KB apart. When that stride is a multiple of 64 KB (k = 4096, 8192:
                 // Mixtral, Qwen3-235B), waves in step hit the same memory channels: measured 5.5 TB/s at k = 8192
                 // and 6.0 at 4096 against 6.5 at 2048; with the rotated start 6.0 and 6.6. Other strides gain
                 // nothing from it (k = 7168: 6.2 either way).
                 a->k % 4096 == 0,
                 scan ? *scan : StreamScan{}, quant ? *quant : StreamQuant{}, nullptr, 0, 0, 0, 0, 0, slots_of(scan, slots)};
  const bool swiglu = a->act == KMOE_ACT_SWIGLU;
  const int live = expected_rows(a->rows, a->rows_hint);
  if (quant) {
    // the down launch of a decode-sized layer: 16 rows per pass, one wave per K range
    KMOE_REQUIRE(!scan && !swiglu && a->variant == 0 && a->row_src == nullptr && !a->acc_out && quant->act &&
                     quant->codes && quant->amax && quant->ld >= a->k && quant->ld % 8 == 0 &&
                     a->k <= kStreamQuantMaxK && a->k / 64 < 24 && ceil_div(live, a->E) <= 10,
                 KMOE_ERR_UNSUPPORTED, "grouped_gemm_i8 (stream): not a launch that can quantise its rows itself");
    // (Four steps of weights in flight and two channel fragments per wave as in the plain launch. Two steps, or one
    // fragment per wave with 2 / 4 / 8 steps - 5 to 6 waves per SIMD - are 1.6 to 3.3 us slower; 6 and 8 steps with
    // two fragments need more registers than four waves per SIMD leave, and this launch needs the four: built for
    // three it took as long as the quantiser's launch and this one together had. Qwen3 decode, layer: 117.5 us with
    // the quantiser's launch, 117.0 built for three waves, 115.1 for four.)
    return launch_stream<Fmt::I8, 1, 2, false, 4, 1, false, true>(p, s);
  }
  if (scan) {
    if (int rc = check_scan(scan, swiglu, a->variant, a->row_src, a->rows)) return rc;
    KMOE_REQUIRE(a->a_rows <= kStreamScanMaxRows, KMOE_ERR_UNSUPPORTED, "grouped_gemm_i8 (stream): %d tokens", a->a_rows);
    return launch_rows16<Fmt::I8, true, true>(p, live, s);
  }
  // a dense matrix: a tail expert alone (activations beyond that kernel's 32-bit offsets stay here)
  if (a->variant == 0 && a->rows == 0 && !swiglu && dense_gemm_i8_reaches(a->a_rows, a->k)) return dense_gemm_i8(a, s);
  // m-fragments per pass from the rows an expert gets under uniform routing
  int mf = a->variant;
  if (mf == 0) {
    // An expert with more rows than one pass holds streams its weights again: leave headroom
    // over the mean for the spread of a random routing (about +-2 sigma at these sizes).
    const int avg = ceil_div(live, a->E);
    mf = avg <= 10 ? 1 : (avg <= 22 ? 2 : (avg <= 48 ? 4 : 8));
  }
  switch (mf) {
    case 1:
      return swiglu ? launch_rows16<Fmt::I8, true, false>(p, live, s)
                    : launch_rows16<Fmt::I8, false, false>(p, live, s);
    case 2:
      return swiglu ? launch_stream<Fmt::I8, 2, 2, true, 4>(p, s) : launch_stream<Fmt::I8, 2, 2, false, 4>(p, s);
    case 4:
      return swiglu ? launch_stream<Fmt::I8, 4, 2, true, 4>(p, s) : launch_stream<Fmt::I8, 4, 2, false, 4>(p, s);
    case 8:
      return swiglu ? launch_stream<Fmt::I8, 8, 2, true, 2>(p, s) : launch_stream<Fmt::I8, 8, 2, false, 2>(p, s);
    default:
      return fail(KMOE_ERR_UNSUPPORTED, "grouped_gemm_i8 (stream): variant=%d must be 0, 1, 2, 4 or 8", a->variant);
  }
}

int stream_gemm_fp8(const kmoe_gemm_fp8_args* a, hipStream_t s, const StreamScan* scan, const StreamSlots* slots) {
  const StreamParams p{reinterpret_cast<const int8_t*>(a->a), a->lda, 128, 0, a->a_scale, a->row_src, a->src_div,
                       reinterpret_cast<const int8_t*>(a->w), a->w_scale, a->lod, a->E, a->n, a->k, a->y, a->ldy, nullptr,
                       reinterpret_cast<const int8_t*>(a->w_tail), a->w_scale_tail, a->tail_row0, a->w_tail ? a->tail_rows : 0,
                       a->tail_src0, a->act_dtype == KMOE_DT_F16, 0, scan ? *scan : StreamScan{}, StreamQuant{},
                       nullptr, 0, 0, 0, 0, 0, slots_of(scan, slots)};
  const bool swiglu = a->act == KMOE_ACT_SWIGLU;
  const int live = expected_rows(a->rows, a->rows_hint);
  if (scan) {
    if (int rc = check_scan(scan, swiglu, a->variant, a->row_src, a->rows)) return rc;
    return launch_rows16<Fmt::F8, true, true>(p, live, s);
  }
  return swiglu ? launch_rows16<Fmt::F8, true, false>(p, live, s) : launch_rows16<Fmt::F8, false, false>(p, live, s);
}

int stream_gemm_bf16(const kmoe_gemm_bf16_args* a, hipStream_t s, const StreamScan* scan, const StreamSlots* slots) {
  const bool half = a->act_dtype == KMOE_DT_F16;
  const StreamSlots columns = slots_of(scan, slots);
  const int live = expected_rows(a->rows, a->rows_hint);
  const StreamParams p{reinterpret_cast<const int8_t*>(a->a), a->lda * 2, 64, 0, nullptr, a->row_src, a->src_div,
                       reinterpret_cast<const int8_t*>(a->w), nullptr, a->lod, a->E, a->n, a->k * 2, a->y, a->ldy, nullptr,
                       nullptr, nullptr, 0, 0, 0, half, 0, scan ? *scan : StreamScan{}, StreamQuant{},
                       nullptr, 0, 0, 0, 0, 0, columns, columns.n == 0 && live < 3ll * a->E};
  const bool swiglu = a->act == KMOE_ACT_SWIGLU;
  if (scan) {
    if (int rc = check_scan(scan, swiglu, a->variant, a->row_src, a->rows)) return rc;
    return half ? launch_rows16<Fmt::F16, true, true>(p, live, s) : launch_rows16<Fmt::BF16, true, true>(p, live, s);
  }
  if (half) return swiglu ? launch_rows16<Fmt::F16, true, false>(p, live, s) : launch_rows16<Fmt::F16, false, false>(p, live, s);
  return swiglu ? launch_rows16<Fmt::BF16, true, false>(p, live, s) : launch_rows16<Fmt::BF16, false, false>(p, live, s);
}

// 16-row launches split K two ways and keep one step (128 values) of loads in flight per wave: fewer registers and more
// waves hide the unpacking and the loads of each other better than a deeper queue does (Qwen3, 64 tokens, layer, steps
// in flight x split: 1x1 81.7 us, 2x1 81.9, 3x1 83.3, 1x2 78.8, 2x2 81.5; Kimi-K2 dimensions, 128 tokens: 1584 / 1577 /
// 1606 / 1568 / 1598).
//
// A gate_up launch of long rows splits K four ways (kW4LongSteps), and so that there are no more workgroups than before, each of which finds its
// rows first, its waves take twice the channels - where that would leave fewer than four for a CU, the same channels. Layers as [hidden x
// intermediate], time over the time with two ways, even load / +2.0 on the logits of eight experts / every token on the same experts:
//   Kimi-K2 dims 2 tokens 0.97 / 0.97 / 0.99, 5 0.95 / 0.95 / 0.95, 12 0.97 / 0.96 / 1.00; 160 of [5120 x 1536], top 6, 3 0.96 / 0.91 / 0.93, 6 0.97 /
//   0.95 / 0.94; 128 of [4096 x 1536], top 8, 5 0.95 / 0.99 / 0.96, 24 1.00 / 0.97 / 0.89; 64 of [4096 x 2048], top 8, 5 0.97 / 1.03 / 1.00, 24 1.01 / 0.95 /
//   0.82; 32 of [4096 x 4096], top 4, 8 1.01 / 1.03 / 0.99, 24 1.01 / 0.95 / 0.90; 256 of [3072 x 512], top 8, 5 0.89 / 0.89 / 0.81.
// Columns of pairs whose expert an earlier column serves ask for their first weights in vain, and twice the channels are twice of them: with many
// workgroups of short work (below 40 and below 28 steps) two ways stay. Four ways there: 128 of [3072 x 4096], top 8, 8 tokens (64 columns of 128
// workgroups) 1.03 / 1.02 / 1.10, 16 (a column per expert) 1.05 / 1.06 / 1.01, 160 of [3072 x 5120], top 6, 10 (60 of 160) 1.02 / 1.02 / 1.09, but 5 (30 of 160)
// 0.99 / 0.98 / 0.98; 128 of [4096 x 6144], top 6, 12 (72 of 192) 1.00 / 1.02 / 1.07, but 5 (30 of 192) 0.97 / 0.98 / 0.97; 64 of [3584 x 8192], top 8, 6 (48 of 256)
// 1.02 / 1.03 / 1.10, but 4 (32 of 256) 0.99 / 0.98 / 0.98. Rows of 2048 values lose 0 to 6 % (Qwen3 dims 7 tokens 41.9 -> 43.1 us, 24 66.0 -> 68.4).
//
// Up to 32 columns of a launch with a column per pair do not fill the chip: gate_up launches keep two steps in flight there (one token 22.5 -> 21.1 and
// 62 -> 59 us), down launches split K four ways (layer: Kimi-K2 dims 2 tokens 0.98 of the time, 3 0.98, 64 of [6144 x 3072], top 4, 3 0.96 / 0.98 / 0.94, but
// 48 columns of Kimi-K2 dims: launch 70.5 -> 74.2 us).
//
// A caller's variant, and rows beyond the reach of the split launches' 32-bit offsets, keep one wave per K range: the tile kernel's order of sums, and
// rows anywhere in memory.
constexpr int kW4LongSteps = 24;  // of 128 values
template <Fmt FMT>
int stream_w4_shape(const StreamParams& p, bool swiglu, bool scan, int passes, bool split, hipStream_t s) {
  const int steps = p.kbytes / 64;
  const long long four_ways = static_cast<long long>(ceil_div(p.n / 2, 32)) * (p.slots.n > 0 ? p.slots.n : p.E);  // workgroups then
  if (passes == 1 && split && swiglu && steps >= kW4LongSteps && (steps >= 40 || four_ways <= (steps >= 28 ? 8192 : 4096))) {
    if (four_ways < 1024)
      return scan ? launch_stream<FMT, 1, 2, true, 1, 4, true>(p, s) : launch_stream<FMT, 1, 2, true, 1, 4>(p, s);
    return scan ? launch_stream<FMT, 1, 4, true, 1, 4, true>(p, s) : launch_stream<FMT, 1, 4, true, 1, 4>(p, s);
  }
  if (passes == 1 && split && p.slots.n > 0 && p.slots.n <= 32)
    return scan ? launch_stream<FMT, 1, 2, true, 2, 2, true>(p, s)
                : (swiglu ? launch_stream<FMT, 1, 2, true, 2, 2>(p, s) : launch_stream<FMT, 1, 2, false, 1, 4>(p, s));
  if (passes == 1 && split)
    return scan ? launch_stream<FMT, 1, 2, true, 1, 2, true>(p, s)
                : (swiglu ? launch_stream<FMT, 1, 2, true, 1, 2>(p, s) : launch_stream<FMT, 1, 2, false, 1, 2>(p, s));
  if (passes == 1) return swiglu ? launch_stream<FMT, 1, 2, true, 1>(p, s) : launch_stream<FMT, 1, 2, false, 1>(p, s);
  if (passes == 2)
    return swiglu ? launch_stream<FMT, 2, 2, true, 2>(p, s) : launch_stream<FMT, 2, 2, false, 2>(p, s);
  return swiglu ? launch_stream<FMT, 4, 2, true, 2>(p, s) : launch_stream<FMT, 4, 2, false, 2>(p, s);
}

int stream_gemm_w4(const kmoe_gemm_w4_args* a, hipStream_t s, int passes, const StreamScan* scan, const StreamSlots* slots,
                   bool rows_fit_32) {
  const int q = a->group_size / 32;
  int shift = -1;
  if ((q & (q - 1)) == 0)
    for (shift = 0; (1 << shift) < q; ++shift) {}
  const int groups = a->k / a->group_size;
  const bool frag16 = a->scale_layout == KMOE_S_FRAG16;
  const bool half = a->act_dtype == KMOE_DT_F16;
  const StreamParams p{reinterpret_cast<const int8_t*>(a->a), a->lda * 2, 256, 0, nullptr, a->row_src, a->src_div,
                       reinterpret_cast<const int8_t*>(a->w), nullptr, a->lod, a->E, a->n, a->k / 2, a->y, a->ldy, nullptr,
                       nullptr, nullptr, 0, 0, 0, half, 0, scan ? *scan : StreamScan{}, StreamQuant{},
                       a->w_scale, groups, frag16 ? 1 : groups, frag16 ? 16 : 1, q, shift, slots_of(scan, slots)};
  const bool swiglu = a->act == KMOE_ACT_SWIGLU;
  if (scan)
    if (int rc = check_scan(scan, swiglu, a->variant, a->row_src, a->rows)) return rc;
  KMOE_REQUIRE(rows_fit_32 || (!scan && !slots), KMOE_ERR_UNSUPPORTED,
               "grouped_gemm_w4a16 (stream): a launch that sorts the pairs itself reaches the activations with 32 bits (rows=%d lda=%lld)",
               a->rows, static_cast<long long>(a->lda));
  const bool split = a->variant == 0 && rows_fit_32;
  return half ? stream_w4_shape<Fmt::W4H>(p, swiglu, scan != nullptr, passes, split, s)
              : stream_w4_shape<Fmt::W4>(p, swiglu, scan != nullptr, passes, split, s);
}

}  // namespace kmoe

using namespace kmoe;

extern "C" int kmoe_tile_weights_i8(const int8_t* src, int8_t* dst, int E, int n, int k, kmoe_stream_t stream) {
  KMOE_REQUIRE(src && dst, KMOE_ERR_NULL, "tile_weights_i8: NULL pointer");
  KMOE_REQUIRE(src != dst, KMOE_ERR_SHAPE, "tile_weights_i8: src and dst must differ (not an in-place transform)");
  KMOE_REQUIRE(E >= 1 && n >= 16 && n % 16 == 0 && k >= 64 && k % 64 == 0, KMOE_ERR_SHAPE,
               "tile_weights_i8: E=%d n=%d k=%d (need n %% 16 == 0, k %% 64 == 0)", E, n, k);
  const long long total_vec = static_cast<long long>(E) * n * k / 16;
  hipLaunchKernelGGL(tile_weights_kernel, dim3(static_cast<unsigned>((total_vec + 255) / 256)), dim3(256), 0,
                     as_stream(stream), src, dst, n, k, total_vec);
  return check_launch("kmoe_tile_weights_i8");
}
