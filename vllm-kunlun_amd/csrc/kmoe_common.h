// Shared device/host helpers for libkmoe (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kmoe.h"

namespace kmoe {

// Rows a launch expects to be live: `rows` bounds the sorted rows (grids and buffers are sized by it), the hint of
// the argument blocks (0: none) says how many of them the caller expects to exist - an expert-parallel share
// sorts only the pairs routed to its own experts. Kernels are CHOSEN by it; every choice is correct for any count.
inline int expected_rows(int rows, int hint) { return hint > 0 && hint < rows ? hint : rows; }

constexpr int kWave = 64;
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// ---- error plumbing (host) -------------------------------------------------
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);
// Compute units of the current device (asked for once).
int compute_units(int* n_cu);
// The calling thread's record of launched GEMM kernels (kmoe_trace_kernels): a launcher notes the kernel it chose.
bool tracing_kernels();
void note_kernel(const char* fmt, ...);
// Writes {0, rows} to lod2: the row offsets of a dense (single-expert) GEMM.
int fill_dense_lod(int32_t* lod2, int rows, hipStream_t stream);
// Weight-streaming int8 GEMM (tiled weights, chunk-major activations); arguments already validated.
// With `scan` (the layer's routed gate_up launch at decode sizes) the launch sorts the routed pairs by expert
// itself: it reads the pairs' expert ids instead of lod / row_src (args->lod and args->row_src are ignored; the
// gather divisor is args->src_div) and leaves what the sort would have left: lod [E+1], expert_m [E],
// moe_index [n_pairs], sorted_src [n_pairs]. Every id must lie in [0, E).
struct StreamScan {
  const int32_t* ids;
  int32_t n_pairs;
  int32_t* lod;
  int32_t* expert_m;
  int32_t* moe_index;
  int32_t* sorted_src;
  int2* slot_rows;  // NULL, or [n_pairs]: a launch with a column of workgroups per pair (pair_scan.h, slots)
};
// The layer's down launch of a batch of few tokens, where the gate_up launch filled slot_rows: columns as there.
struct StreamSlots {
  const int32_t* ids;
  const int2* rows;
  int32_t n;  // 0: a column per expert
};
constexpr int kStreamSlotMaxPairs = 256;
constexpr int kStreamScanMaxPairs = 4096;
constexpr int kStreamScanMaxRows = 512;  // tokens: no expert gets more rows than that
// With `quant` (the layer's down launch at decode sizes, k <= kStreamQuantMaxK) the launch quantises its rows
// itself: it reads them as bf16 / half values (act, row stride ld; args->act_dtype) instead of args->a / a_max and
// leaves codes (chunk-major [k/64][args->a_rows][64]) and row maxes where the quantiser's launch would have.
struct StreamQuant {
  const uint16_t* act;
  int64_t ld;
  int8_t* codes;
  float* amax;
};
constexpr int kStreamQuantMaxK = 1024;
// Second quantisation, down projection and combine of a layer of a few tokens in one launch (few_tokens.hip). Rows of
// act: routed pairs by moe_index, then (w_tail) the M rows of a shared expert of the same width. Tiled weights.
struct FewDown {
  int32_t M, K, H, I;
  int32_t kbytes;  // bytes of a weight row
  const int32_t *ids, *moe_index;
  const float* topk_w;
  const uint16_t* act;  // [rows, I]
  int32_t rows;
  int8_t* codes;  // what the quantiser's launch would leave: codes (int8: chunk-major) and row maxes / group scales
  float* code_aux;
  const int8_t* w;
  const float* w_aux;
  const int8_t* w_tail;
  const float* w_aux_tail;
  const uint16_t* w_scale;  // 4-bit: as in StreamParams
  int32_t groups, s_ch, s_g, gs32, gs_shift;
  uint16_t* down;  // [rows, H]
  float out_scale, shared_scale;
  uint16_t* out;  // [M, H]
  int32_t f16;
};
constexpr int kFewMaxI = 2048, kFewMaxWaves = 16;  // K, and one for the shared expert
int few_down(const FewDown& p, int format, hipStream_t stream);
// Dense int8 GEMM of a few rows (a tail expert alone, tiled weights, chunk-major activations); arguments already validated.
int dense_gemm_i8(const kmoe_gemm_i8_args* args, hipStream_t stream);
bool dense_gemm_i8_reaches(int a_rows, int k);  // whether its 32-bit offsets reach these activations
int stream_gemm_i8(const kmoe_gemm_i8_args* args, hipStream_t stream, const StreamScan* scan, const StreamQuant* quant,
                   const StreamSlots* slots);
// The same kernel on fp8 block-scaled and on 16-bit weights (tiled; row-major activations).
int stream_gemm_fp8(const kmoe_gemm_fp8_args* args, hipStream_t stream, const StreamScan* scan, const StreamSlots* slots);
int stream_gemm_bf16(const kmoe_gemm_bf16_args* args, hipStream_t stream, const StreamScan* scan, const StreamSlots* slots);
// kmoe_grouped_gemm_* with the options above for the layer's own launches.
int grouped_gemm_i8_checked(const kmoe_gemm_i8_args* args, kmoe_stream_t stream, const StreamScan* scan,
                            const StreamQuant* quant, const StreamSlots* slots);
int grouped_gemm_fp8_checked(const kmoe_gemm_fp8_args* args, kmoe_stream_t stream, const StreamScan* scan,
                             const StreamSlots* slots);
int grouped_gemm_bf16_checked(const kmoe_gemm_bf16_args* args, kmoe_stream_t stream, const StreamScan* scan,
                              const StreamSlots* slots);
// Whether a launch of these dimensions on tiled weights and without a variant runs on the weight-streaming kernel:
// up to 10 rows per expert (the tile kernel's cross-over, measured for all formats), rows of the lengths it takes.
constexpr int kStreamMaxRows = 10;
inline bool streams_fp8(int live_rows, int E, int k) { return ceil_div(live_rows, E) <= kStreamMaxRows && k <= 8192; }
inline bool streams_bf16(int live_rows, int E, int k) { return ceil_div(live_rows, E) <= kStreamMaxRows && k % 32 == 0; }
// kmoe_grouped_gemm_w4a16 with `scan` for the layer's routed gate_up launch where it runs on the streaming kernel
// (w4_gate_up_streams says whether a launch of these dimensions does). a_rows: rows of the activations, every source row
// lies below (-1: not known).
int grouped_gemm_w4a16_checked(const kmoe_gemm_w4_args* args, kmoe_stream_t stream, const StreamScan* scan,
                               const StreamSlots* slots, long long a_rows);
// The streaming kernel on packed 4-bit weights; passes: 1, 2, 4 for 16, 32, 64 rows per pass; rows_fit_32: 32-bit
// offsets reach every source row.
int stream_gemm_w4(const kmoe_gemm_w4_args* args, hipStream_t stream, int passes, const StreamScan* scan,
                   const StreamSlots* slots, bool rows_fit_32);
bool w4_gate_up_streams(int rows, int rows_hint, long long tokens, int E, int n, int k);
// Whether a 32-bit byte offset reaches every value of `rows` 16-bit activation rows (and a row's worth beyond, what the
// kernels' K steps add to the offset of a row).
inline bool w4_rows_fit_32(long long rows, int64_t lda, int k) {
  return lda < (1ll << 31) && static_cast<uint64_t>(rows) * static_cast<uint64_t>(lda) * 2u + static_cast<uint64_t>(k) * 2u < (1ull << 32);
}
// Persistent 128-row-tile GEMMs for many rows per expert (tiled weights, row-major activations);
// arguments already validated.
int tiled_gemm_i8(const kmoe_gemm_i8_args* args, hipStream_t stream);
int tiled_gemm_fp8(const kmoe_gemm_fp8_args* args, hipStream_t stream);
int tiled_gemm_bf16(const kmoe_gemm_bf16_args* args, hipStream_t stream);
// The router logits as a routing kernel finds them: f32, or 16-bit values (bf16 / half: what a gate that is an
// ordinary 16-bit Linear leaves; widening them is exact, so reading them where they are used instead of after a
// conversion launch changes no bit), or the partial planes of a split-K router GEMM, `plane_stride` floats apart.
struct LogitsView {
  const void* p;
  int planes;  // > 1: f32 partial sums; the logit is their sum, plane 0 first
  size_t plane_stride;
  int type;  // 0: f32, 1: bf16, 2: half (planes == 1)
};
struct RouteArgs {
  LogitsView logits;  // [M, E]
  const float* bias;
  int M, E, K, renorm, n_group, topk_group;
  float scale;
  float* topk_w;
  int32_t* topk_ids;
};
// Routing, first quantisation, sort and gate_up projection of a layer of up to kFewRouted tokens and 64 pairs in one launch
// (few_tokens.hip); leaves topk_w / topk_ids, what the sort would leave, and act.
struct FewGateUp {
  RouteArgs route;
  int32_t H, I, kbytes;
  const uint16_t* x;  // [M, H]
  const int8_t* w;    // [E, 2 I, H] tiled
  const float* w_aux;
  const int8_t* w_tail;
  const float* w_aux_tail;
  const uint16_t* w_scale;  // 4-bit: as in StreamParams
  int32_t groups, s_ch, s_g, gs32, gs_shift;
  StreamScan sort;  // what the sort would leave, slot_rows too (ids and n_pairs are not looked at)
  uint16_t* act;  // [P (+ M), I]
  int32_t f16;
  int32_t alone, alone_at;  // (the launcher's) one token whose row waves 1 to 3 bring to LDS, this far in
};
constexpr int kFewRouted = 4;
constexpr int kFewRowBytes = 25 * 1024;  // of LDS for the rows of a launch: five workgroups on a CU
int few_gate_up(const FewGateUp& p, int format, bool sigmoid, hipStream_t stream);
// The checks of the routing arguments (and n_group <= 1 made one group).
int check_route(RouteArgs* r, bool sigmoid);
// Routing of M tokens and, for KMOE_FMT_INT8 / _FP8_BLOCK where the kernel takes the row length, the quantisation of
// x [M,H] in the same launch (*quantised says whether it was). M >= 1.
int route_and_quantise(RouteArgs r, bool sigmoid, int format, const uint16_t* x, int H, void* xq, float* x_aux,
                       bool chunked, bool f16, bool* quantised, hipStream_t stream);

// Router GEMM pieces for the fused layer: the split (ks planes, mf*16 tokens per wave) chosen for
// a shape, and the launch that leaves the partial planes [ks][M][E] (ks == 1: the logits).
void router_plan(int M, int H, int E, int* ks_out, int* mf_out);
int router_gemm_planes(const uint16_t* x, int64_t ld_x, const uint16_t* w, int M, int H, int E, float* planes,
                       size_t plane_stride, int64_t ld_out, int ks, int mf, hipStream_t stream, bool f16 = false);
// out[m,e] = planes[0][m,e] + planes[1][m,e] + ... (that order); out may be plane 0 itself.
int router_reduce(const float* planes, size_t plane_stride, int n_planes, int M, int E, float* out, int64_t ld_out,
                  hipStream_t stream);

#define KMOE_REQUIRE(cond, code, ...) \
  do {                                \
    if (!(cond)) return ::kmoe::fail((code), __VA_ARGS__); \
  } while (0)

// ---- bf16 <-> f32, bit-exact round-to-nearest-even --------------------------
__host__ __device__ inline float bf16_to_f32(uint16_t h) {
  union { uint32_t u; float f; } v;
  v.u = static_cast<uint32_t>(h) << 16;
  return v.f;
}

__host__ __device__ inline uint16_t f32_to_bf16(float f) {
  union { uint32_t u; float f; } v;
  v.f = f;
  uint32_t u = v.u;
  if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

// Device-only: the gfx950 conversion instruction (v_cvt_pk_bf16_f32, round to nearest
// even) — same bits as f32_to_bf16 for every finite input, one instruction per pair.
typedef float kmoe_v2f __attribute__((ext_vector_type(2)));
typedef __bf16 kmoe_v2bf __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pack2_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((kmoe_v2f){lo, hi}, kmoe_v2bf));
}
__device__ inline uint16_t f32_to_bf16_hw(float f) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f)); }

// ---- activation dtype: bf16 or IEEE half, chosen per call (a wave-uniform flag) ----------
// Both are 16-bit patterns in uint16_t tensors. Conversions are round-to-nearest-even; a value
// beyond the half range becomes infinity, as in every IEEE conversion.
__device__ inline float half_to_f32(uint16_t h) { return static_cast<float>(__builtin_bit_cast(_Float16, h)); }
// (The empty asm keeps the f32 value as it is: without it the compiler folds a preceding f32 multiplication into
// a mixed-precision instruction that rounds the exact product to half ONCE, which differs from rounding it to
// f32 first - the sequence the result contract fixes - whenever the f32 rounding lands on a half tie.)
__device__ inline uint16_t f32_to_half(float f) {
  asm("" : "+v"(f));
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
}
__device__ inline float act_to_f32(uint16_t h, bool f16) { return f16 ? half_to_f32(h) : bf16_to_f32(h); }
__device__ inline uint16_t f32_to_act(float f, bool f16) { return f16 ? f32_to_half(f) : f32_to_bf16(f); }
typedef _Float16 kmoe_v2h __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pack2_half(float lo, float hi) {
  asm("" : "+v"(lo));
  asm("" : "+v"(hi));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((kmoe_v2f){lo, hi}, kmoe_v2h));
}

// ---- fixed-sequence transcendental -----------------------------------------
// exp(x) as one fixed sequence of IEEE single operations (mul, round-to-even,
// fma, exact power-of-two scaling), so that a CPU restatement performing the
// same sequence gives the same bits. Argument clamped to [-86, 86] so neither
// the result nor 1/(1+result) leaves the normal range. Error < 2 ulp.
__device__ inline float exp_fixed(float x) {
  x = fminf(fmaxf(x, -86.0f), 86.0f);
  const float n = __builtin_rintf(x * 0x1.715476p+0f);            // x * log2(e)
  float r = __builtin_fmaf(n, -0x1.62e4p-1f, x);                  // - n * ln2_hi
  r = __builtin_fmaf(n, -0x1.7f7d1cp-20f, r);                     // - n * ln2_lo
  float p = 0x1.a01a02p-13f;                                      // 1/5040
  p = __builtin_fmaf(p, r, 0x1.6c16c2p-10f);                      // 1/720
  p = __builtin_fmaf(p, r, 0x1.111112p-7f);                       // 1/120
  p = __builtin_fmaf(p, r, 0x1.555556p-5f);                       // 1/24
  p = __builtin_fmaf(p, r, 0x1.555556p-3f);                       // 1/6
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return __builtin_ldexpf(p, static_cast<int>(n));
}

__device__ inline float sigmoid_fixed(float x) { return 1.0f / (1.0f + exp_fixed(-x)); }

// ---- SiLU of the GEMM epilogues ----------------------------------------------
// silu(g) = g / (1 + e^-g) on the hardware's transcendental unit: v_exp_f32 (2^t) and v_rcp_f32, each within
// one ulp, five instructions in all - the fixed-sequence exp and an IEEE divide cost thirty and were a sixth of
// the prefill gate_up launch. The two instructions are not correctly rounded, so no CPU sequence gives their
// bits; but SiLU is only ever applied to a 16-BIT activation value (gate is rounded to bf16 / half first, as the
// reference's silu_and_mul reads a 16-bit tensor), i.e. to one of 65536 arguments per activation type:
// kmoe_silu_table writes this function's result for every one of them, which is how a checker follows it bit
// for bit. Every kernel calls THIS function, so a token's result does not depend on the kernel that computes it.
// Arguments below -87 count as -87 (1 + 2^t and its reciprocal stay in the normal range; the result there,
// -1.4e-36, is 0 for every purpose, also for g = -inf, which would otherwise give inf x 0).
__device__ inline float silu_hw(float g) {
  const float gc = fmaxf(g, -87.0f);
  const float d = 1.0f + __builtin_amdgcn_exp2f(gc * -0x1.715476p+0f);  // 1 + 2^(-g log2(e))
  return gc * __builtin_amdgcn_rcpf(d);
}
// gpt-oss activation on a (gate, up) pair of bf16 values, one rounding at the end:
// g = min(gate, limit), u = clamp(up, -limit, limit), out = (u + 1) * g * sigmoid(alpha * g)
// (reference: swigluoai_and_mul, ops/_custom_ops.py:728-742).
__device__ inline uint16_t swigluoai_bf16(uint16_t gate, uint16_t up, float alpha, float limit) {
  const float g = fminf(bf16_to_f32(gate), limit);
  const float u = fminf(fmaxf(bf16_to_f32(up), -limit), limit);
  const float glu = g * sigmoid_fixed(g * alpha);
  return f32_to_bf16((u + 1.0f) * glu);
}

// ---- wave64 helpers ---------------------------------------------------------
__device__ inline int lane_id() { return static_cast<int>(threadIdx.x) & (kWave - 1); }

// Reductions over a wave or groups of its lanes stay on the vector unit: exchanges between halves and rows (v_permlane32_swap,
// v_permlane16_swap), then moves inside the rows of 16 lanes (DPP) - a chain of some twelve instructions where six exchanges
// through the LDS crossbar (__shfl_xor) are six round trips of it. A token's routing waits for two of them: its maximum
// 0.40 -> 0.20 us, exponentials and sum 0.40 -> 0.28.
// Lane l gets lane (l - N) mod 16 of its row: between lanes whose groups of 2 N already agree, the same as lane l ^ N.
template <int N>
__device__ inline uint32_t row_rotated(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x120 + N, 0xf, 0xf, true));
}
// op of every lane's value and that of lane l ^ 16 / l ^ 32 (the two operands in the same order in both lanes)
template <class Op>
__device__ inline uint32_t across_rows(uint32_t v, Op op) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // even rows twice, odd rows twice
  return op(r[0], r[1]);
}
template <class Op>
__device__ inline uint32_t across_halves(uint32_t v, Op op) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // lower half twice, upper half twice
  return op(r[0], r[1]);
}
// op over aligned groups of G lanes (16, 32 or 64), in every lane; an op that rounds sees the tree t[l] = t[l] op t[l ^ off],
// off = G/2 ... 1, whose steps take the same two numbers on both sides.
template <int G, class Op>
__device__ inline uint32_t group_reduce(uint32_t v, Op op) {
  static_assert(G == 16 || G == 32 || G == 64, "whole rows of 16 lanes");
  if constexpr (G > 32) v = across_halves(v, op);
  if constexpr (G > 16) v = across_rows(v, op);
  v = op(v, row_rotated<8>(v));
  v = op(v, row_rotated<4>(v));
  v = op(v, row_rotated<2>(v));
  return op(v, row_rotated<1>(v));
}
template <class Op>
__device__ inline auto on_floats(Op op) {
  return [op](uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, op(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)));
  };
}
template <int G>
__device__ inline float group_max(float v) {
  return __builtin_bit_cast(float, group_reduce<G>(__builtin_bit_cast(uint32_t, v), on_floats([](float a, float b) { return fmaxf(a, b); })));
}
__device__ inline float wave_max(float v) { return group_max<kWave>(v); }
template <int G>
__device__ inline uint32_t group_max_u32(uint32_t v) {
  return group_reduce<G>(v, [](uint32_t a, uint32_t b) { return max(a, b); });
}
// Sum over the wave, the same bits in every lane: the balanced tree of group_reduce.
__device__ inline float wave_sum_tree(float v) {
  return __builtin_bit_cast(float, group_reduce<kWave>(__builtin_bit_cast(uint32_t, v), on_floats([](float a, float b) { return a + b; })));
}

__device__ inline int wave_sum_int(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// A float as an unsigned int with the same order (-0 counts as +0). Never 0, which stands for "not a candidate" where
// the largest is picked: one NaN pattern (all bits set, what memory filled with -1 holds) would map there and counts as
// its neighbour instead; no number does.
__host__ __device__ inline uint32_t ordered_bits(float v) {
  union { float f; uint32_t u; } b;
  b.f = v + 0.0f;
  const uint32_t key = (b.u & 0x80000000u) ? ~b.u : (b.u | 0x80000000u);
  return key != 0 ? key : 1;
}
__device__ inline uint64_t lanemask_lt() {
  return (static_cast<uint64_t>(1) << lane_id()) - 1;
}

inline hipStream_t as_stream(kmoe_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

}  // namespace kmoe
