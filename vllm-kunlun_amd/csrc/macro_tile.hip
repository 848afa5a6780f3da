// Grouped GEMM on tiles of up to 192 rows x 256 weight rows with BOTH operands staged in LDS; tiled weights, int8
// (v_mfma_i32_16x16x64_i8), 16-bit operands (v_mfma_f32_16x16x32_bf16 / _f16) and block-scaled fp8 (v_mfma_scale_f32_16x16x128_f8f6f4).
//
// One workgroup per CU, persistent: eight waves, two along the rows (every other fragment of 16 rows each) and four along the
// channels (64 each), 6 x 4 accumulator fragments a wave. Activations and weights come global -> LDS by asynchronous copies, once
// per CU, and from there into two register sets: one feeds the MFMAs of a step (64 bytes of K), the other is read for the next step.
//   activations  128 bytes of K per row and chunk (two steps), three chunk buffers, rows gathered through the sort, swizzled as in
//                tiled_gemm.hip (vector c of row r at position c ^ r % 8); rows past the tile's end are not fetched
//   weights      16 KB per step, five step buffers; an expert's weights pass the caches where it has one tile (see MacroParams::past)
// Steps are numbered through all tiles of a workgroup: the copies of the next tile's first steps leave during the last steps of this
// one, so the rings never drain between tiles. A finished tile is dequantised during the next one's first step, fragment by fragment
// as that step's MFMAs take its accumulators over, and stored during that tile's first six steps: stored at once, by all CUs at about
// the same time, the results cost their whole write time (Qwen3 dims, down, 8192 tokens, 268 MB: 155 us, without the stores 98).
// What bounds it: the bytes, where experts have few rows (DeepSeek-V3 dims, int8, gate_up, 47 rows: 7.5 GB in 1150 us, 6.6 TB/s, where
// the tiles of tiled_gemm.hip, whose weights go through registers, take 1285); with many rows the copies into LDS (Qwen3 dims, int8,
// gate_up, 8192 tokens: 219 us; without the MFMAs 162, from hot weights 200) and the matrix unit (1.9 POP/s there, 243 us and
// 1.7 before). Tiles of 256 rows (whose registers and LDS leave no room for the third chunk buffer and the late stores): 225 us, down
// 147 against 139; K begun at a step of its own per channel block: 0 to -2 %, -8 % on [4096 x 7168]; tile heights chosen by the rows
// of each launch (96 to 192): 0.
//
// Waits. A wave's copies complete in issue order, and its stores count among them. At an odd step s a wave issues the activation
// chunk of steps s + 5 and s + 6, then the weights of step s + 5; at an even one the weights alone. At the top of step s everything
// older than what left after the weights of step s + 1 (at step s - 4) has landed; the barrier behind the wait publishes it, and says
// that every wave holds its fragments of step s, whose buffers the copies issued behind it may overwrite.
// fp8 runs chunk by chunk (see chunk_f8): registers for one set of fragments beside the partial sums, six weight buffers, and two
// chunk buffers - or, where 128 rows hold nearly every expert, three and tiles of 128 rows (DeepSeek-V3 dims, gate_up, 94 rows 1338 ->
// 1286 us). Its copies leave together behind the chunk's first LDS requests (one after each MFMA group: 1354, these 1276).
// All LDS accesses of the pipeline are assembly statements: one that the compiler sees would wait for every copy in flight.
#include <utility>

#include "buffer_ops.h"
#include "kmoe_common.h"
#include "macro_tile.h"

namespace kmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kMWaves = 8, kMThreads = kMWaves * kWave;
constexpr int kMWaveCols = 4;              // waves along the channels
constexpr int kMFrags = 4;                 // channel fragments of a wave
constexpr int kMWeightStep = 16 * 1024;    // bytes of weights per step: 16 fragments of 16 channels x 64 bytes of K
constexpr int kMChunk = 128;               // bytes of K per activation row and chunk

template <class F, int... I>
__device__ __forceinline__ void m_for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void m_for(F&& f) {
  m_for_each(f, std::make_integer_sequence<int, N>{});
}

enum class MOp { I8, BF16, F16, F8 };

// The four MFMAs of row fragment I, left out if the tile has no rows there (a branch the compiler does not see: the K loop
// stays one basic block). FIRST: the sums begin here.
template <MOp OP, bool FIRST, int I>
__device__ __forceinline__ void m_mfma4(v4i (&c)[4], const v4i (&w)[4], const v4i& a, int live) {
#define KMOE_M_SKIP "s_cmp_le_i32 %[live], %[i]\n\ts_cbranch_scc1 1f\n\t"
#define KMOE_M_MORE(X)                                                                                       \
  asm volatile(KMOE_M_SKIP X " %[c0], %[w0], %[a], %[c0]\n\t" X " %[c1], %[w1], %[a], %[c1]\n\t" X             \
                             " %[c2], %[w2], %[a], %[c2]\n\t" X " %[c3], %[w3], %[a], %[c3]\n1:"                \
               : [c0] "+v"(c[0]), [c1] "+v"(c[1]), [c2] "+v"(c[2]), [c3] "+v"(c[3])                            \
               : [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]), [a] "v"(a), [live] "s"(live), \
                 [i] "n"(I)                                                                                  \
               : "scc")
#define KMOE_M_FIRST(X)                                                                                      \
  asm volatile(KMOE_M_SKIP X " %[c0], %[w0], %[a], 0\n\t" X " %[c1], %[w1], %[a], 0\n\t" X                     \
                             " %[c2], %[w2], %[a], 0\n\t" X " %[c3], %[w3], %[a], 0\n1:"                       \
               : [c0] "=&v"(c[0]), [c1] "=&v"(c[1]), [c2] "=&v"(c[2]), [c3] "=&v"(c[3])                        \
               : [w0] "v"(w[0]), [w1] "v"(w[1]), [w2] "v"(w[2]), [w3] "v"(w[3]), [a] "v"(a), [live] "s"(live), \
                 [i] "n"(I)                                                                                  \
               : "scc")
#define KMOE_M_BOTH(X)                \
  if constexpr (FIRST) KMOE_M_FIRST(X); \
  else KMOE_M_MORE(X)
  if constexpr (OP == MOp::I8) {
    KMOE_M_BOTH("v_mfma_i32_16x16x64_i8");
  } else if constexpr (OP == MOp::BF16) {
    KMOE_M_BOTH("v_mfma_f32_16x16x32_bf16");
  } else {
    KMOE_M_BOTH("v_mfma_f32_16x16x32_f16");
  }
#undef KMOE_M_SKIP
#undef KMOE_M_MORE
#undef KMOE_M_FIRST
#undef KMOE_M_BOTH
}

// LDS reads without the compiler's waits (see above), and the wait that makes a register set usable
template <int OFF>
__device__ __forceinline__ void m_read(v4i& v, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void m_request_f32(float& v, uint32_t addr) {
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
}
__device__ __forceinline__ void m_landed(v4i (&w)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
}
// at most N younger LDS operations in flight: these have landed
template <int N>
__device__ __forceinline__ void m_wait8(v4i& lo, v4i& hi) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo), "+v"(hi) : "n"(N) : "memory");
}
template <int MF>
__device__ __forceinline__ void m_landed_a(v4i (&a)[MF]) {
#pragma unroll
  for (int i = 0; i < MF; ++i) asm volatile("" : "+v"(a[i]));
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t) const_cast<void*>(p)));
}
__device__ __forceinline__ float m_read_f32(uint32_t addr) {
  float v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(addr) : "memory");
  return v;
}
__device__ __forceinline__ int m_read_i32(uint32_t addr) {
  int v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(addr) : "memory");
  return v;
}

// A buffer descriptor over `bytes` from base, as assembly takes it.
__device__ __forceinline__ v4i m_rsrc(const void* base, uint32_t bytes) {
  const uint64_t addr = reinterpret_cast<uint64_t>(base);
  return (v4i){static_cast<int>(addr), static_cast<int>((addr >> 32) & 0xffffu), static_cast<int>(bytes), 0x00020000};
}
// 1 KB of weights global -> LDS, asynchronously: lane l's 16 bytes land at `to` + 16 l. Past the caches or not (buffer_ops.h) is a bit of the
// instruction, so there are two of it and a branch that the compiler does not see (the step stays one basic block).
// A vector-memory instruction may read a scalar register five wait states after a vector instruction wrote it - which reloads of
// spilled ones do - and the compiler keeps that distance for its own instructions only: five stand in front of each load here.
__device__ __forceinline__ void m_copy_weights(const int8_t* base, uint32_t lane_off, uint32_t at, uint32_t to, int past) {
  const v4i rsrc = m_rsrc(base, 0xffffffffu);
  uint32_t keep;  // (the compiler takes m0 for its own)
  asm volatile(
      "s_mov_b32 %[keep], m0\n\t"
      "s_mov_b32 m0, %[to]\n\t"
      "s_nop 0\n\t"
      "s_cmp_eq_u32 %[past], 0\n\t"
      "s_cbranch_scc1 1f\n\t"
      "buffer_load_dwordx4 %[lo], %[r], %[at] offen nt lds\n\t"
      "s_branch 2f\n"
      "1:\n\t"
      "buffer_load_dwordx4 %[lo], %[r], %[at] offen lds\n"
      "2:\n\t"
      "s_mov_b32 m0, %[keep]"
      : [keep] "=&s"(keep)
      : [to] "s"(to), [past] "s"(past), [lo] "v"(lane_off), [r] "s"(rsrc), [at] "s"(at)
      : "scc", "memory");
}

// Sixteen bytes of results a lane, past the caches or not, likewise. (The wait states keep a vector instruction behind it from
// overwriting the results before the store has read them; those in front are the distance that m_copy_weights keeps.)
// "Past" is non-temporal for the gate_up launch's rows (SHORT), and for the down launch's, several times as many, written through
// the L2 as they come (sc1): DeepSeek-V3 dims, layer, us, non-temporal / written through: int8, 700 tokens 1884 / 1863, 2048 2093 / 2080, 4096
// 2478 / 2465; fp8, 1200 1937 / 1914, 3001 2380 / 2376 (down launch 732 -> 710 at 2048, combine 63 -> 51; the gate_up launch's rows written through:
// 1262 -> 1301).
template <bool SHORT>
__device__ __forceinline__ void m_store(const v4i& v, const v4i& rsrc, uint32_t at, int past) {
  if constexpr (SHORT)
    asm volatile(
        "s_nop 2\n\t"
        "s_cmp_eq_u32 %[past], 0\n\t"
        "s_cbranch_scc1 1f\n\t"
        "buffer_store_dwordx4 %[v], %[at], %[r], 0 offen nt\n\t"
        "s_branch 2f\n"
        "1:\n\t"
        "buffer_store_dwordx4 %[v], %[at], %[r], 0 offen\n"
        "2:\n\t"
        "s_nop 1"
        :
        : [v] "v"(v), [at] "v"(at), [r] "s"(rsrc), [past] "s"(past)
        : "scc", "memory");
  else
    asm volatile(
        "s_nop 2\n\t"
        "s_cmp_eq_u32 %[past], 0\n\t"
        "s_cbranch_scc1 1f\n\t"
        "buffer_store_dwordx4 %[v], %[at], %[r], 0 offen sc1\n\t"
        "s_branch 2f\n"
        "1:\n\t"
        "buffer_store_dwordx4 %[v], %[at], %[r], 0 offen\n"
        "2:\n\t"
        "s_nop 1"
        :
        : [v] "v"(v), [at] "v"(at), [r] "s"(rsrc), [past] "s"(past)
        : "scc", "memory");
}
// Rows of each of an expert's mt tiles: split evenly in whole fragments (an expert with more tiles than a tile has fragments
// keeps full ones: the rounding could leave the last one without rows).
template <int TM>
__device__ __forceinline__ int split_rows(int rows, int mt) {
  return mt <= TM / 16 ? ((rows + mt - 1) / max(mt, 1) + 15) & ~15 : TM;
}
constexpr int kMItems = 32;               // items resolved at a time

struct MTile {
  int it, e, row0, nb, end;
  int past;  // its weights are read once: past the caches
  bool valid;
};

// OP: operands; F16: the results are IEEE half; MF: row fragments of a wave (tiles of 32 MF rows), 6; fp8 also 4.
template <MOp OP, bool SWIGLU, bool F16, int MF>
__global__ __launch_bounds__(kMThreads, 1) void macro_tile_kernel(const MacroParams p) {
  constexpr bool I8 = OP == MOp::I8, F8 = OP == MOp::F8;
  constexpr int kWeightSlots = F8 ? 6 : 5, kChunkBufs = F8 && MF > 4 ? 2 : 3;  // (the copies and waits below are written for these)
  constexpr int kTM = 32 * MF;
  constexpr int NFH = SWIGLU ? kMFrags / 2 : kMFrags;  // output fragments of a wave
  constexpr int kNA = MF / 2;                          // copies per wave and activation chunk: 8 rows (1 KB) each
  constexpr int kABytes = kTM * kMChunk;
  __shared__ __attribute__((aligned(1024))) int8_t ring_a[kChunkBufs][kABytes];
  __shared__ __attribute__((aligned(1024))) int8_t ring_w[kWeightSlots][kMWeightStep];
  // per tile parity: the tile's channel and row absmax values, divided by 127 in place at its start
  __shared__ __attribute__((aligned(16))) float sw_lds[I8 ? 2 : 1][I8 ? 256 : 4];
  __shared__ __attribute__((aligned(16))) float sa_lds[I8 ? 2 : 1][I8 ? kTM : 4];
  // fp8: the row scales of four chunks, two groups of chunks in turn; per tile parity the scales of its two blocks of 128 channels
  __shared__ __attribute__((aligned(16))) float asc_lds[F8 ? 2 : 1][F8 ? 4 * kTM : 4];
  __shared__ __attribute__((aligned(16))) float wsc_lds[F8 ? 2 : 1][F8 ? 2 * kMacroBlocks : 4];
  __shared__ __attribute__((aligned(16))) int idx_lds[kTM];  // gather entries of the next tile's rows
  __shared__ int items[4][kMItems];
  extern __shared__ int m_dyn[];
  static_assert(sizeof(ring_a) + sizeof(ring_w) + sizeof(sw_lds) + sizeof(sa_lds) + sizeof(asc_lds) + sizeof(wsc_lds) + sizeof(idx_lds) + sizeof(items) + kMacroTables <= 160 * 1024, "LDS of a CU");
  const int n_exp = p.E + (p.w_tail ? 1 : 0);
  int* row_lo = m_dyn;              // [E + 1]: lod
  int* tile_lo = m_dyn + p.E + 1;   // [n_exp + 1]: first m-tile of each expert, then the total

  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 3, wm = wave >> 2;
  const int li = lane & 15, lg = lane >> 4;
  const int n_half = SWIGLU ? p.n / 2 : p.n;
  const int ksteps = p.k / 64;
  auto rows_begin = [&](int e) { return e < p.E ? row_lo[e] : p.tail_row0; };
  auto rows_end = [&](int e) { return e < p.E ? row_lo[e + 1] : p.tail_row0 + p.tail_rows; };

  // ---- rows and m-tiles of every expert ----
  for (int e = threadIdx.x; e <= p.E; e += kMThreads) row_lo[e] = p.lod[e];
  __syncthreads();
  if (wave == 0) {
    int carry = 0;
    for (int base = 0; base < n_exp; base += kWave) {
      const int e = base + lane;
      const int mine = e < n_exp ? (rows_end(e) - rows_begin(e) + kTM - 1) / kTM : 0;
      int incl = mine;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const int o = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += o;
      }
      if (e < n_exp) tile_lo[e] = carry + incl - mine;
      carry += __shfl(incl, kWave - 1, kWave);
    }
    if (lane == 0) tile_lo[n_exp] = carry;
  }
  __syncthreads();
  // ---- the workgroup's items, as in tiled_gemm.hip: the list of (m-tile, channel block) pairs, expert by expert, in eight
  // segments, one per XCD, which the workgroups of the XCD walk side by side; an expert's rows split evenly over its m-tiles. (A tail
  // expert's items, which the list ends with, shared out over the XCDs: DeepSeek-V3 dims, layer, even load / +2.0 on the logits of eight experts, time
  // over this order's, int8 2048 tokens 0.99 / 0.99, 4096 1.00 / 1.02, 5000 1.00 / 1.02, but 256 experts of [4096 x 1024], top 8, 2048 1.01 / 1.03, 128 of
  // [5120 x 1536], top 8, 2048 1.00 / 1.03, 64 of [4096 x 1408], top 6, 2048 1.00 / 1.07.) ----
  const int n_items = tile_lo[n_exp] * p.n_blocks;
  const int seg = (n_items + 7) >> 3;
  const int xcd = blockIdx.x & 7;
  const int seg_end = min((xcd + 1) * seg, n_items);
  const int per_xcd = gridDim.x >> 3;  // gridDim.x is a multiple of 8
  auto resolve_items = [&](int it0) {
    if (wave == 0 && lane < kMItems) {
      const int lid = xcd * seg + (blockIdx.x >> 3) + (it0 + lane) * per_xcd;
      int e = -1, row0 = 0, nb = 0, end = 0, past = 0;
      if (lid < seg_end) {
        const int m_tile = lid / p.n_blocks;
        int lo = 0, hi = n_exp - 1;  // the last e with tile_lo[e] <= m_tile
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (tile_lo[mid] <= m_tile) lo = mid;
          else hi = mid - 1;
        }
        e = lo;
        const int first = tile_lo[e], mt = tile_lo[e + 1] - first;
        const int u = lid - first * p.n_blocks;
        int m;
        if (p.m_major) {
          m = u / p.n_blocks;
          nb = u - m * p.n_blocks;
        } else {
          nb = u / mt;
          m = u - nb * mt;
        }
        const int rows_e = rows_end(e) - rows_begin(e);
        const int stride = split_rows<kTM>(rows_e, mt);
        row0 = rows_begin(e) + m * stride;
        past = p.past && mt == 1;
        end = min(rows_end(e), row0 + stride);
      }
      items[0][lane] = e;
      items[1][lane] = row0;
      items[2][lane] = 2 * nb + past;
      items[3][lane] = end;
    }
    __syncthreads();
  };
  resolve_items(0);
  auto find_tile = [&](int it) -> MTile {
    if (it > 0 && (it & (kMItems - 1)) == 0) resolve_items(it);
    MTile t{it, 0, 0, 0, 0, 0, false};
    const uint32_t at = lds_addr(&items[0][0]) + 4u * (it & (kMItems - 1));
    int e, row0, nb, end;
    asm volatile(
        "ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:%5\n\tds_read_b32 %2, %4 offset:%6\n\tds_read_b32 %3, %4 offset:%7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(e), "=&v"(row0), "=&v"(nb), "=&v"(end)
        : "v"(at), "n"(4 * kMItems), "n"(8 * kMItems), "n"(12 * kMItems)
        : "memory");
    t.e = __builtin_amdgcn_readfirstlane(e);
    t.valid = t.e >= 0;
    t.row0 = __builtin_amdgcn_readfirstlane(row0);
    nb = __builtin_amdgcn_readfirstlane(nb);
    t.nb = nb >> 1;
    t.past = nb & 1;
    t.end = __builtin_amdgcn_readfirstlane(end);
    return t;
  };
  MTile cur = find_tile(0);
  if (!cur.valid) return;  // (the whole workgroup; nothing is in flight)

  // ---- loads ----
  constexpr uint32_t kRange = 0xfffffff0u;  // an offset of kRange lies outside every descriptor here: nothing is read
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.a), 0, kRange, 0x00020000);
  const uint32_t lane16 = lane * 16u;
  // What is computed from this is computed where it is used. fp8 without SiLU-mul, whose late results take twice the registers: addresses
  // held through the tile loop were spilled, and each reload waited for all copies in flight (Qwen3 dims, down, 512 rows per expert
  // 185 -> 167 us, DeepSeek-V3 dims, 170 931 -> 907, 512 2408 -> 2339). The other instances have the registers, and hold them.
  constexpr bool kTight = F8 && !SWIGLU && MF == 6;
  auto here = [](uint32_t v) __attribute__((always_inline)) -> uint32_t {
    if constexpr (kTight) asm volatile("" : "+v"(v));
    return v;
  };
  auto lane_here = [&]() __attribute__((always_inline)) -> int { return kTight ? static_cast<int>(here(lane16) >> 4) : lane; };
  // channel of fragment f of the waves in column c (0: past the last channel, never stored)
  auto col_of = [&](const MTile& t, int c, int f, bool& ok) -> int {
    const int fh = SWIGLU ? f % NFH : f;
    const int ch = (t.nb * kMWaveCols + c) * NFH * 16 + fh * 16;
    ok = ch < n_half;
    return (SWIGLU && f >= NFH) ? n_half + ch : ch;
  };
  struct Weights {  // where a tile's weights lie: the expert's, and this wave's two fragments of every step
    const int8_t* base;
    uint32_t off0, off1;
    int past;
  };
  auto weights_of = [&](const MTile& t) -> Weights {
    Weights w;
    w.base = t.e >= p.E ? p.w_tail : p.w + static_cast<size_t>(t.e) * p.n * p.k;
    bool ok0, ok1;
    const int c0 = col_of(t, (2 * wave) >> 2, (2 * wave) & 3, ok0), c1 = col_of(t, (2 * wave) >> 2, (2 * wave + 1) & 3, ok1);
    w.past = t.past;
    w.off0 = static_cast<uint32_t>(ok0 ? c0 / 16 : 0) * ksteps * 1024u;
    w.off1 = static_cast<uint32_t>(ok1 ? c1 / 16 : 0) * ksteps * 1024u;
    return w;
  };
  // copy h (0, 1) of a step's weights
  auto dma_w = [&](const Weights& w, int step, uint32_t slot_at, int h) __attribute__((always_inline)) {
    m_copy_weights(w.base, lane16, (h ? w.off1 : w.off0) + static_cast<uint32_t>(step) * 1024u,
                   __builtin_amdgcn_readfirstlane(lds_addr(&ring_w[0][0])) + slot_at + wave * 2048u + h * 1024u, w.past);
  };
  uint32_t a_off[kNA];
  // copy i of this wave fills rows 8 (kNA wave + i) + lane / 8 of a chunk buffer
  auto dma_row = [&]() __attribute__((always_inline)) { return wave * 8 * kNA + (lane_here() >> 3); };
  auto dma_a = [&](int chunk, uint32_t buf_at, int i) __attribute__((always_inline)) {
    buffer_load16_to_lds(a_rsrc, (lds_ptr_t)(&ring_a[0][0] + buf_at + (wave * kNA + i) * 1024), a_off[i],
                         static_cast<uint32_t>(chunk) * kMChunk);
  };
  // sorted row r of tile t (past its end: its first), and the row of p.a that `fetched`, the row's gather entry, names
  auto clamp_row = [&](const MTile& t, int r) { return r < t.end ? r : t.row0; };
  auto src_row = [&](const MTile& t, int rr, int fetched) -> uint32_t {
    const bool gathered = t.e < p.E && p.row_src != nullptr;
    const uint32_t entry = static_cast<uint32_t>(fetched);
    const uint32_t divided = p.div_magic ? __umulhi(entry, p.div_magic) : entry;  // entry / src_div
    return gathered ? divided : static_cast<uint32_t>(rr + (t.e >= p.E ? p.tail_src0 - p.tail_row0 : 0));
  };
  // the tile's absmax values into the slots of its scales: waves 0-3 its rows', waves 4-7 its channels'
  auto dma_scales = [&](const MTile& t, int parity, int fetched) __attribute__((always_inline)) {
    if constexpr (I8) {
      if (wave < 4) {
        if (64 * wave < kTM)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(p.a_max), (lds_ptr_t)&sa_lds[parity][64 * wave], 4,
                                                   src_row(t, clamp_row(t, t.row0 + 64 * wave + lane), fetched) * 4u, 0, 0, 0);
      } else {
        bool ok;
        const int c = col_of(t, wave - 4, lane >> 4, ok);
        const float* w_max = t.e >= p.E ? p.w_max_tail : p.w_max + static_cast<size_t>(t.e) * p.n;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(w_max), (lds_ptr_t)&sw_lds[parity][64 * (wave - 4)], 4,
                                                 static_cast<uint32_t>(ok ? c + li : 0) * 4u, 0, 0, 0);
      }
    }
  };
  auto scales_in_place = [&](int parity) __attribute__((always_inline)) {
    if constexpr (I8) {
      static_assert(kTM % kWave == 0 && kTM <= 256, "whole waves bring the rows' values");
      if (64 * wave >= kTM && wave < 4) return;
      const uint32_t at = wave < 4 ? lds_addr(&sa_lds[parity][threadIdx.x]) : lds_addr(&sw_lds[parity][threadIdx.x - 256]);
      const float scaled = m_read_f32(at) / 127.0f;
      asm volatile("ds_write_b32 %0, %1" : : "v"(at), "v"(scaled) : "memory");
    }
  };

  // ---- fragment reads: step j of a chunk takes vector 4 j + lg of every row ----
  uint32_t fa[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    fa[j] = lds_addr(&ring_a[0][0]) + static_cast<uint32_t>((wm * 16 + li) * kMChunk + (((4 * j + lg) ^ (li & 7)) << 4));
  const uint32_t fw = lds_addr(&ring_w[0][0]) + wn * 4096u + lane16;
  v4i af[2][MF], wf[2][kMFrags];
  v4i acc[MF][kMFrags];

  // ---- first tile ----
  auto row_offset = [&](const MTile& t, int i, int fetched) -> uint32_t {  // rows past the tile's end are not read
    const int r = t.row0 + dma_row() + 8 * i;
    const int l = lane_here();
    const uint32_t a_col = static_cast<uint32_t>((l & 7) ^ ((l >> 3) & 7)) * 16u;  // vector c of row r at position c ^ r % 8
    return r < t.end ? src_row(t, r, fetched) * static_cast<uint32_t>(p.lda) + a_col : kRange;  // < 4 GiB: host-checked
  };
  Weights w_cur = weights_of(cur);
#pragma unroll
  for (int i = 0; i < kNA; ++i)
    a_off[i] = row_offset(cur, i, (p.row_src && cur.e < p.E) ? p.row_src[clamp_row(cur, cur.row0 + dma_row() + 8 * i)] : 0);
  {
    const int rr = clamp_row(cur, cur.row0 + 64 * (wave & 3) + lane);
    const int fetched = (p.row_src && cur.e < p.E) ? p.row_src[rr] : 0;
    __builtin_amdgcn_sched_barrier(0);
    dma_scales(cur, 0, fetched);
  }
  // fp8: a row's scales of four chunks from block `base` on; the tile's weight scales
  const int kblocks = p.k / 128;
  uint32_t asc_off = 0;  // the scales of tile row 64 wave + lane (waves 0-2)
  auto dma_row_scales = [&](int base, int group) __attribute__((always_inline)) {
    if constexpr (F8) {
      if (64 * wave < kTM)
        buffer_load16_to_lds(make_rsrc(p.a_max), (lds_ptr_t)&asc_lds[group][256 * wave], asc_off, static_cast<uint32_t>(base) * 4u);
    }
  };
  auto dma_tile_scales = [&](const MTile& t, int parity, int fetched) __attribute__((always_inline)) {
    if constexpr (F8) {
      asc_off = src_row(t, clamp_row(t, t.row0 + 64 * (wave & 3) + lane_here()), fetched) * static_cast<uint32_t>(kblocks) * 4u;
      const int b = wave - 4;  // waves 4 and 5: a block of 128 channels each
      if (b == 0 || b == 1) {
        const int row = SWIGLU ? t.nb + b * (n_half / 128) : min(2 * t.nb + b, p.n / 128 - 1);
        const float* ws = t.e >= p.E ? p.w_max_tail : p.w_max + static_cast<size_t>(t.e) * (p.n / 128) * kblocks;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(ws), (lds_ptr_t)&wsc_lds[parity][b * kMacroBlocks], 4,
                                                 static_cast<uint32_t>(row * kblocks + min(lane_here(), kblocks - 1)) * 4u, 0, 0, 0);
      }
    }
  };
  if constexpr (F8) {
    const int fetched = (p.row_src && cur.e < p.E) ? p.row_src[clamp_row(cur, cur.row0 + 64 * (wave & 3) + lane)] : 0;
    __builtin_amdgcn_sched_barrier(0);
    dma_tile_scales(cur, 0, fetched);
    dma_row_scales(0, 0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {  // in the order of the chunks -2 and -1
#pragma unroll
      for (int i = 0; i < kNA; ++i)
        if (kChunkBufs == 3 || c == 1) dma_a(kChunkBufs == 3 ? c : 0, kChunkBufs == 3 ? c * kABytes : 0, i);
#pragma unroll
      for (int st = 2 * c; st < 2 * c + 2; ++st) {
        dma_w(w_cur, st, st * kMWeightStep, 0);
        dma_w(w_cur, st, st * kMWeightStep, 1);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  } else {
  // in the order of the steps -5 to -1
#pragma unroll
  for (int st = 0; st < 5; ++st) {
    if (st % 2 == 0) {
#pragma unroll
      for (int i = 0; i < kNA; ++i) dma_a(st / 2, st / 2 * kABytes, i);
    }
    dma_w(w_cur, st, st * kMWeightStep, 0);
    dma_w(w_cur, st, st * kMWeightStep, 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  vmem_wait<2 * kNA + 6>();  // steps 0 and 1 and the first chunk
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  m_for<MF>([&](auto i) __attribute__((always_inline)) { m_read<i * 32 * kMChunk>(af[0][i], fa[0]); });
  m_for<kMFrags>([&](auto f) __attribute__((always_inline)) { m_read<f * 1024>(wf[0][f], fw); });
  m_landed(wf[0]);
  m_landed_a(af[0]);
  }

  uint32_t slot = 0;      // bytes: the weight slot of this step; the next one's follows it
  uint32_t buf = 0;       // bytes: the buffer of this step's chunk
  int live = 0;

  // ---- the results of the tile before: finished during step 0, stored during steps 0 to 5 ----
  constexpr int kPairs = NFH / 2;     // 64-byte pieces of a row a wave holds
  constexpr int kStores = MF * kPairs;
  constexpr int kStoreSteps = F8 ? (MF == 4 ? 2 : 3) : 6;  // (fp8: chunks)
  static_assert(kStores % kStoreSteps == 0, "the same number of stores in each of the first steps");
  constexpr int kPerStep = kStores / kStoreSteps;
  v4i done[MF][kPairs];
  v4i y_rsrc = m_rsrc(p.y, 0);  // (nothing yet: stores nothing)
  uint32_t y_off = 0;
  int live_done = 0;
  float sa[MF];
  v4i sw_raw[kMFrags];
  const uint32_t ld_bytes = static_cast<uint32_t>(p.ldy) * 2u;
  auto take_scales = [&](int parity) __attribute__((always_inline)) {
    if constexpr (I8) {
      const uint32_t sa_at = lds_addr(&sa_lds[parity][wm * 16 + li]);
      const uint32_t sw_at = lds_addr(&sw_lds[parity][wn * 64 + lg * 4]);
      m_for<MF>([&](auto i) __attribute__((always_inline)) { m_request_f32<i * 128>(sa[i], sa_at); });
      m_for<kMFrags>([&](auto f) __attribute__((always_inline)) { m_read<f * 64>(sw_raw[f], sw_at); });
      m_landed(sw_raw);
#pragma unroll
      for (int i = 0; i < MF; ++i) asm volatile("" : "+v"(sa[i]));
    }
  };
  auto finish = [&](auto i_tag) __attribute__((always_inline)) {  // row fragment i: dequantise, SiLU-mul, round
    constexpr int i = decltype(i_tag)::value;
    auto value = [&](int f, int q) -> float {
      if constexpr (I8) return (static_cast<float>(acc[i][f][q]) * sa[i]) * __builtin_bit_cast(v4f, sw_raw[f])[q];
      else return __builtin_bit_cast(v4f, acc[i][f])[q];
    };
    uint2 out[NFH];
#pragma unroll
    for (int f = 0; f < NFH; ++f) {
      float y[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        y[q] = value(f, q);
        if constexpr (SWIGLU) {  // gate and up are 16-bit values first
          const float u = value(f + NFH, q);
          const float g = F16 ? half_to_f32(f32_to_half(y[q])) : bf16_to_f32(f32_to_bf16_hw(y[q]));
          y[q] = silu_hw(g) * (F16 ? half_to_f32(f32_to_half(u)) : bf16_to_f32(f32_to_bf16_hw(u)));
        }
      }
      out[f] = F16 ? make_uint2(pack2_half(y[0], y[1]), pack2_half(y[2], y[3])) : make_uint2(pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3]));
    }
    // A lane holds 4 channels of each fragment; exchanged between the rows of 16 lanes, 8 of one fragment: lanes lg = 0 to 3
    // then cover the 64 bytes of two fragments' channels of their row.
#pragma unroll
    for (int h = 0; h < kPairs; ++h) {
      const auto x = __builtin_amdgcn_permlane16_swap(out[2 * h].x, out[2 * h + 1].x, false, false);
      const auto y = __builtin_amdgcn_permlane16_swap(out[2 * h].y, out[2 * h + 1].y, false, false);
      done[i][h] = (v4i){static_cast<int>(x[0]), static_cast<int>(y[0]), static_cast<int>(x[1]), static_cast<int>(y[1])};
    }
  };
  // where a finished tile's results go: rows past its end lie outside the descriptor, channels past the last get an offset that does
  auto aim = [&](const MTile& t) __attribute__((always_inline)) {
    const int rows = min(t.end - t.row0, kTM);
    y_rsrc = m_rsrc(p.y + static_cast<size_t>(t.row0) * p.ldy, static_cast<uint32_t>(rows - 1) * ld_bytes + static_cast<uint32_t>(n_half) * 2u);
    live_done = live;
  };
  int y_col = 0;
  auto store = [&](auto n_tag) __attribute__((always_inline)) {  // store n of the tile before
    constexpr int n = decltype(n_tag)::value;
    constexpr int i = n / kPairs, h = n % kPairs;
    const uint32_t at = y_col + 32 * h < n_half ? y_off + static_cast<uint32_t>(i * 32) * ld_bytes + 64u * h : kRange;
    m_store<SWIGLU>(done[i][h], y_rsrc, at, p.y_past);
  };

  // One step: its fragments are in registers (set S), the next step's are read into the other set. a_chunk (odd steps): the
  // activation chunk to copy; w, w_step: the weights. One copy leaves after each of the first MFMA groups: all of them at once,
  // by eight waves, kept the last wave waiting for its turn while its MFMAs could run (232 -> 225 us at 256 rows). Steps 0 to 5
  // also store what step 0 finished.
  [[maybe_unused]] auto step = [&](auto st_tag, int a_chunk, const Weights& w, int w_step, auto start) __attribute__((always_inline)) {
    constexpr int st = decltype(st_tag)::value;  // 0-5: steps of a tile that store; beyond: its parity and whether stores may be in flight
    constexpr bool odd = st & 1, first = st == 0;
    constexpr int S = odd ? 1 : 0;
    __builtin_amdgcn_sched_barrier(0);
    // younger than the weights of step s + 1, which left at s - 4 (as did, before them at an odd s, the chunk of s + 1): the
    // copies of s - 3 to s - 1, and the stores of s - 4 to s - 1
    constexpr int kStored = [] {
      int n = 0;
      for (int t = st - 4; t < st; ++t) n += t >= 0 && t < kStoreSteps;
      return n;
    }();
    vmem_wait<(odd ? 1 : 2) * kNA + 6 + kStored * kPerStep>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    start();
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t w_to = slot, a_to = buf;
    slot = slot + kMWeightStep == kWeightSlots * kMWeightStep ? 0 : slot + kMWeightStep;
    if constexpr (odd) buf = buf + kABytes == kChunkBufs * kABytes ? 0 : buf + kABytes;
    const uint32_t a_at = fa[odd ? 0 : 1] + buf, w_at = fw + slot;
    m_for<MF>([&](auto i) __attribute__((always_inline)) {
      m_read<i * 32 * kMChunk>(af[S ^ 1][i], a_at);
      if constexpr (i < kMFrags) m_read<i * 1024>(wf[S ^ 1][i], w_at);
      if constexpr (first) {
        if (i < live_done) finish(i);
      }
      m_mfma4<OP, first, i>(acc[i], wf[S], af[S][i], live);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (odd) {
        if constexpr (i < kNA) dma_a(a_chunk, a_to, i);
        else if constexpr (i < kNA + 2) dma_w(w, w_step, w_to, i - kNA);
      } else {
        if constexpr (i == 1 || i == 3) dma_w(w, w_step, w_to, i >> 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (st < kStoreSteps) m_for<kPerStep>([&](auto n) __attribute__((always_inline)) { store(std::integral_constant<int, st * kPerStep + n>{}); });
    m_landed(wf[S ^ 1]);
    m_landed_a(af[S ^ 1]);
  };
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  constexpr std::integral_constant<int, 2> s2{};
  constexpr std::integral_constant<int, 3> s3{};
  constexpr std::integral_constant<int, 4> s4{};
  constexpr std::integral_constant<int, 5> s5{};
  constexpr std::integral_constant<int, 10> even{};
  constexpr std::integral_constant<int, 11> odd{};
  auto nothing = [] {};
  static_assert(F8 ? kStoreSteps <= 3 : kStoreSteps == 6, "steps written out below");

  // fp8: one whole chunk. An MFMA covers its 128 bytes of K - the two 1 KB weight blocks are its two halves, and the activation
  // fragment takes the same two - and one weight scale each: its partial sum is scaled and added in f32. The fragments of a chunk
  // are read while it runs, so a buffer is free one chunk later than above: at its start chunk c copies the activations of
  // c + kChunkBufs - 1 and the weights of c + 2. The scaling of fragment n - 1 follows the MFMAs of fragment n.
  int group = 0;  // of asc_lds: that of this chunk
  [[maybe_unused]] auto chunk_f8 = [&](auto st_tag, int c, int parity, int a_chunk, const Weights& w, int w_chunk, auto start) __attribute__((always_inline)) {
    if constexpr (F8) {
      constexpr int st = decltype(st_tag)::value;
      constexpr bool first = st == 0;
      __builtin_amdgcn_sched_barrier(0);
      // younger than chunk c's operands: the weights of c + 1 and c - 1's stores; with three buffers, whose activations left before
      // c's weights, the activations of c + 1 and c - 2's stores, too
      constexpr int kStored = (st >= 1 && st - 1 < kStoreSteps ? 1 : 0) + (kChunkBufs == 3 && st >= 2 && st - 2 < kStoreSteps ? 1 : 0);
      vmem_wait<4 + (kChunkBufs == 3 ? kNA : 0) + kStored * kPerStep>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      start();
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t a_to = buf == 0 ? (kChunkBufs - 1) * kABytes : buf - kABytes;
      const uint32_t w_to = slot >= 2 * kMWeightStep ? slot - 2 * kMWeightStep : slot + 4 * kMWeightStep;
      const uint32_t a_lo = fa[0] + buf, a_hi = kTight ? a_lo ^ 64u : fa[1] + buf;  // (bit 2 of the vector's position)
      const uint32_t w_at = kTight ? lds_addr(&ring_w[0][0]) + wn * 4096u + slot + here(lane16) : fw + slot;
      const int base = min(c & ~3, kblocks - 4);
      const uint32_t sa_at = lds_addr(&asc_lds[0][0]) + static_cast<uint32_t>(group * 16 * kTM + (wm * 16 + (lane_here() & 15)) * 16 + 4 * (c - base));
      const uint32_t sw_at = lds_addr(&wsc_lds[parity][SWIGLU ? 0 : (wn >> 1) * kMacroBlocks]) + 4u * c;
      float sw[2], sa_c[2], sc[2][2];
      v4i lo[2], hi[2], wl[kMFrags], wh[kMFrags];
      v4f blk[2][kMFrags];
      auto request = [&](auto n_tag) __attribute__((always_inline)) {
        constexpr int n = decltype(n_tag)::value;
        m_read<n * 32 * kMChunk>(lo[n & 1], a_lo);
        m_read<n * 32 * kMChunk>(hi[n & 1], a_hi);
        m_request_f32<n * 512>(sa_c[n & 1], sa_at);
      };
      auto multiply = [&](int n, int f) __attribute__((always_inline)) {
        v8i av, wv;
        av.lo = lo[n & 1], av.hi = hi[n & 1];
        wv.lo = wl[f], wv.hi = wh[f];
        blk[n & 1][f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv, av, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
      };
      auto add = [&](auto n_tag) __attribute__((always_inline)) {
        constexpr int n = decltype(n_tag)::value;
#pragma unroll
        for (int f = 0; f < kMFrags; ++f) {
          v4f sum = __builtin_bit_cast(v4f, acc[n][f]);
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[q] = __builtin_fmaf(blk[n & 1][f][q], sc[n & 1][SWIGLU ? f / 2 : 0], first ? 0.0f : sum[q]);
          acc[n][f] = __builtin_bit_cast(v4i, sum);
        }
      };
      m_request_f32<0>(sw[0], sw_at);
      if constexpr (SWIGLU) m_request_f32<4 * kMacroBlocks>(sw[1], sw_at);
      request(std::integral_constant<int, 0>{});
      m_for<kMFrags>([&](auto f) __attribute__((always_inline)) {
        m_read<f * 1024>(wl[f], w_at);
        m_read<kMWeightStep + f * 1024>(wh[f], w_at);
      });
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kNA; ++i) dma_a(a_chunk, a_to, i);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        dma_w(w, 2 * w_chunk + i, w_to + i * kMWeightStep, 0);
        dma_w(w, 2 * w_chunk + i, w_to + i * kMWeightStep, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      m_for<MF>([&](auto n) __attribute__((always_inline)) {
        if constexpr (n == 0) {
          m_wait8<6>(wl[0], wh[0]);
          asm volatile("" : "+v"(lo[0]), "+v"(hi[0]), "+v"(sa_c[0]), "+v"(sw[0]));
          if constexpr (SWIGLU) asm volatile("" : "+v"(sw[1]));
          request(std::integral_constant<int, 1>{});
          m_wait8<7>(wl[1], wh[1]);
          m_wait8<5>(wl[2], wh[2]);
          m_wait8<3>(wl[3], wh[3]);
        } else {
          if constexpr (n + 1 < MF) {
            request(std::integral_constant<int, n + 1>{});
            m_wait8<3>(lo[n & 1], hi[n & 1]);
          } else {
            m_wait8<0>(lo[n & 1], hi[n & 1]);
          }
          asm volatile("" : "+v"(sa_c[n & 1]));
        }
        if constexpr (first) {
          if (n < live_done) finish(n);
        }
        if (n < live) {  // (wave-uniform)
#pragma unroll
          for (int f = 0; f < kMFrags; ++f) multiply(n, f);
          sc[n & 1][0] = sa_c[n & 1] * sw[0];
          if constexpr (SWIGLU) sc[n & 1][1] = sa_c[n & 1] * sw[1];
        }
        if constexpr (n > 0) {
          if (n - 1 < live) add(std::integral_constant<int, n - 1>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if (MF - 1 < live) add(std::integral_constant<int, MF - 1>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (st < kStoreSteps) m_for<kPerStep>([&](auto n) __attribute__((always_inline)) { store(std::integral_constant<int, st * kPerStep + n>{}); });
      buf = buf + kABytes == kChunkBufs * kABytes ? 0 : buf + kABytes;
      slot = slot + 2 * kMWeightStep == kWeightSlots * kMWeightStep ? 0 : slot + 2 * kMWeightStep;
    }
  };

  for (int parity = 0;; parity ^= 1) {
    const MTile nxt = find_tile(cur.it + 1);
    const MTile look = nxt.valid ? nxt : cur;  // (after the last tile its first steps are copied again: the waits count copies)
    {
      const int rows = cur.end - cur.row0;
      live = __builtin_amdgcn_readfirstlane(max(0, min(MF, (rows - 16 * wm + 31) >> 5)));
    }
    auto fetch_next = [&]() __attribute__((always_inline)) {  // the gather entries of the next tile's rows
      if (p.row_src && 64 * wave < kTM && wave < 4) {
        const int rr = clamp_row(look, look.row0 + 64 * wave + lane_here());
        __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(p.row_src), (lds_ptr_t)&idx_lds[64 * wave], 4,
                                                 static_cast<uint32_t>(look.e < p.E ? rr : 0) * 4u, 0, 0, 0);
      }
    };
    auto next_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kNA; ++i) a_off[i] = row_offset(look, i, m_read_i32(lds_addr(&idx_lds[dma_row() + 8 * i])));
      return m_read_i32(lds_addr(&idx_lds[min(64 * (wave & 3) + lane_here(), kTM - 1)]));
    };
    const Weights w_nxt = weights_of(look);
    if constexpr (F8) {
      auto group_of = [&](int c) { return min(c, kblocks - 4); };
      if (cur.it > 0) group ^= 1;  // (copied during the tile before)
      constexpr int ahead = kChunkBufs - 1;
      chunk_f8(s0, 0, parity, ahead, w_cur, 2, fetch_next);
      chunk_f8(s1, 1, parity, 1 + ahead, w_cur, 3, nothing);
      chunk_f8(s2, 2, parity, 2 + ahead, w_cur, 4, [&]() __attribute__((always_inline)) { dma_row_scales(group_of(4), group ^ 1); });
      for (int c = 3; c < kblocks - 2; ++c) {
        if ((c & 3) == 0) group ^= 1;
        chunk_f8(even, c, parity, c + ahead, w_cur, c + 2, [&]() __attribute__((always_inline)) {
          if ((c & 3) == 2 && c + 2 < kblocks) dma_row_scales(group_of(c + 2), group ^ 1);
        });
      }
      // the last two: the copies go over to the next tile
      if (((kblocks - 2) & 3) == 0) group ^= 1;
      chunk_f8(even, kblocks - 2, parity, ahead == 2 ? 0 : kblocks - 1, w_nxt, 0, [&]() __attribute__((always_inline)) {
        if constexpr (ahead == 2) dma_tile_scales(look, parity ^ 1, next_rows());
      });
      if (((kblocks - 1) & 3) == 0) group ^= 1;
      chunk_f8(even, kblocks - 1, parity, ahead - 1, w_nxt, 1, [&]() __attribute__((always_inline)) {
        if constexpr (ahead == 1) dma_tile_scales(look, parity ^ 1, next_rows());
        dma_row_scales(0, group ^ 1);
      });
    } else {
    step(s0, 0, w_cur, 5, [&]() __attribute__((always_inline)) {
      fetch_next();
      scales_in_place(parity);
    });
    step(s1, 3, w_cur, 6, nothing);
    step(s2, 0, w_cur, 7, nothing);
    step(s3, 4, w_cur, 8, nothing);
    step(s4, 0, w_cur, 9, nothing);
    step(s5, 5, w_cur, 10, nothing);
    for (int ks = 6; ks < ksteps - 6; ks += 2) {
      step(even, 0, w_cur, ks + 5, nothing);
      step(odd, (ks >> 1) + 3, w_cur, ks + 6, nothing);
    }
    // the last six: the copies go over to the next tile
    step(even, 0, w_cur, ksteps - 1, [&]() __attribute__((always_inline)) {  // (the gather entries landed before the wait of an odd step before)
      dma_scales(look, parity ^ 1, next_rows());
    });
    step(odd, 0, w_nxt, 0, nothing);
    step(even, 0, w_nxt, 1, nothing);
    step(odd, 1, w_nxt, 2, nothing);
    step(even, 0, w_nxt, 3, nothing);
    step(odd, 2, w_nxt, 4, nothing);
    }

    // the MFMAs came from assembly statements, so the compiler knows of no wait for their results
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    take_scales(parity);
    aim(cur);
    y_col = (cur.nb * kMWaveCols + wn) * NFH * 16 + (lg & 1) * 16 + (lg >> 1) * 8;
    y_off = static_cast<uint32_t>(wm * 16 + li) * ld_bytes + static_cast<uint32_t>(y_col) * 2u;
    if (!nxt.valid) break;
    cur = nxt;
    w_cur = w_nxt;
  }
  m_for<MF>([&](auto i) __attribute__((always_inline)) {
    if (i < live_done) finish(i);
  });
  m_for<kStores>([&](auto n) __attribute__((always_inline)) { store(n); });
  vmem_wait<0>();  // no copy may land in LDS that is another workgroup's by then
}

template <MOp OP, bool SWIGLU, bool F16, int MF>
int launch_macro(MacroParams p, int rows, hipStream_t s, int n_cu, const char* what) {
  constexpr int NFH = SWIGLU ? 2 : 4;
  const int n_exp = p.E + (p.w_tail ? 1 : 0);
  p.n_blocks = ceil_div(SWIGLU ? p.n / 2 : p.n, kMWaveCols * NFH * 16);
  const int max_tiles = (rows + p.tail_rows) / (32 * MF) + min(n_exp, rows + p.tail_rows);
  const long long max_items = static_cast<long long>(p.n_blocks) * max_tiles;
  const int grid = static_cast<int>(min((max_items + 7) / 8 * 8, static_cast<long long>(ceil_div(n_cu, 8) * 8)));
  const size_t dyn = sizeof(int) * (static_cast<size_t>(p.E) + 1 + n_exp + 1);
  if (tracing_kernels())
    note_kernel("macro_tile_kernel<%s%s, %s, %dx256 tile, both operands through LDS>", OP == MOp::I8 ? "int8" : (OP == MOp::F8 ? "fp8" : (OP == MOp::F16 ? "f16" : "bf16")),
                ((OP == MOp::I8 || OP == MOp::F8) && F16) ? " -> f16" : "", SWIGLU ? "SiLU-mul" : "plain", 32 * MF);
  hipLaunchKernelGGL((macro_tile_kernel<OP, SWIGLU, F16, MF>), dim3(grid), dim3(kMThreads), dyn, s, p);
  return check_launch(what);
}

}  // namespace

int macro_tile(const MacroParams& p, int kind, bool swiglu, bool f16, int rows, hipStream_t s, int n_cu, const char* what) {
  if (kind == 2) {
    if (p.low) {
      if (f16) return swiglu ? launch_macro<MOp::F8, true, true, 4>(p, rows, s, n_cu, what) : launch_macro<MOp::F8, false, true, 4>(p, rows, s, n_cu, what);
      return swiglu ? launch_macro<MOp::F8, true, false, 4>(p, rows, s, n_cu, what) : launch_macro<MOp::F8, false, false, 4>(p, rows, s, n_cu, what);
    }
    if (f16) return swiglu ? launch_macro<MOp::F8, true, true, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::F8, false, true, 6>(p, rows, s, n_cu, what);
    return swiglu ? launch_macro<MOp::F8, true, false, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::F8, false, false, 6>(p, rows, s, n_cu, what);
  }
  if (kind == 0) {
    if (f16) return swiglu ? launch_macro<MOp::I8, true, true, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::I8, false, true, 6>(p, rows, s, n_cu, what);
    return swiglu ? launch_macro<MOp::I8, true, false, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::I8, false, false, 6>(p, rows, s, n_cu, what);
  }
  if (f16) return swiglu ? launch_macro<MOp::F16, true, true, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::F16, false, true, 6>(p, rows, s, n_cu, what);
  return swiglu ? launch_macro<MOp::BF16, true, false, 6>(p, rows, s, n_cu, what) : launch_macro<MOp::BF16, false, false, 6>(p, rows, s, n_cu, what);
}

}  // namespace kmoe
