// Host side of libkmoe: error state, and the fused layer call that strings the
// stage kernels together on one stream out of one caller-owned workspace.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "asked_once.h"
#include "few_rows.h"
#include "kmoe_common.h"
#include "macro_tile.h"

namespace kmoe {

static thread_local char g_error[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
  return code;
}

// ---- record of the GEMM kernels a thread launches (kmoe_trace_kernels) ----
static thread_local bool g_trace_on = false;
static thread_local char g_trace[4096] = "";
static thread_local size_t g_trace_len = 0;

bool tracing_kernels() { return g_trace_on; }
void note_kernel(const char* fmt, ...) {
  if (!g_trace_on || g_trace_len + 2 >= sizeof(g_trace)) return;
  va_list ap;
  va_start(ap, fmt);
  const int n = vsnprintf(g_trace + g_trace_len, sizeof(g_trace) - g_trace_len - 1, fmt, ap);
  va_end(ap);
  if (n < 0) return;
  g_trace_len = g_trace_len + static_cast<size_t>(n) < sizeof(g_trace) - 2 ? g_trace_len + static_cast<size_t>(n)
                                                                           : sizeof(g_trace) - 2;
  g_trace[g_trace_len++] = '\n';
  g_trace[g_trace_len] = '\0';
}

int compute_units(int* n_cu) {
  static AskedOnce found;
  const int count = found.get([] {
    int dev = 0, n = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess ? n : 0;
  });
  if (count < 1) return fail(KMOE_ERR_LAUNCH, "cannot query the device");
  *n_cu = count;
  return KMOE_OK;
}

int check_launch(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err == hipSuccess) return KMOE_OK;
  return fail(KMOE_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(err));
}

}  // namespace kmoe

using namespace kmoe;

extern "C" const char* kmoe_last_error(void) { return g_error; }
extern "C" const char* kmoe_version(void) { return "kmoe 0.3 gfx950"; }
extern "C" void kmoe_trace_kernels(int on) {
  if (on) {
    g_trace[0] = '\0';
    g_trace_len = 0;
  }
  g_trace_on = on != 0;
}
extern "C" const char* kmoe_traced_kernels(void) { return g_trace; }

namespace {

// formats whose GEMMs read the bf16 activations themselves (no activation quantisation)
bool bf16_activations(int format) { return format == KMOE_FMT_BF16 || format == KMOE_FMT_W4A16; }

int check_shape(const kmoe_moe_args* a) {
  KMOE_REQUIRE(a, KMOE_ERR_NULL, "moe_forward: args is NULL");
  KMOE_REQUIRE(a->M >= 0 && a->H >= 16 && a->E >= 1 && a->K >= 1 && a->I >= 16, KMOE_ERR_SHAPE,
               "moe_forward: M=%d H=%d E=%d K=%d I=%d", a->M, a->H, a->E, a->K, a->I);
  KMOE_REQUIRE(a->format == KMOE_FMT_INT8 || a->format == KMOE_FMT_FP8_BLOCK || a->format == KMOE_FMT_BF16 ||
                   a->format == KMOE_FMT_W4A16,
               KMOE_ERR_UNSUPPORTED, "moe_forward: format=%d unknown", a->format);
  if (a->format == KMOE_FMT_W4A16) {
    KMOE_REQUIRE(a->I_shared == 0, KMOE_ERR_UNSUPPORTED, "moe_forward: no shared expert with 4-bit weights");
    KMOE_REQUIRE(a->w_layout == KMOE_W_TILED, KMOE_ERR_UNSUPPORTED, "moe_forward: 4-bit weights must be tiled");
    KMOE_REQUIRE(a->group_size >= 32 && a->group_size % 32 == 0 && a->H % a->group_size == 0 &&
                     a->I % a->group_size == 0,
                 KMOE_ERR_SHAPE, "moe_forward: group_size=%d must be a multiple of 32 dividing H=%d and I=%d",
                 a->group_size, a->H, a->I);
  }
  const int mult = a->format == KMOE_FMT_FP8_BLOCK || a->format == KMOE_FMT_W4A16 ? 128 : 16;
  KMOE_REQUIRE(a->H % mult == 0 && a->I % mult == 0, KMOE_ERR_SHAPE,
               "moe_forward: H=%d and I=%d must be multiples of %d", a->H, a->I, mult);
  const int Eg = a->E_global > 0 ? a->E_global : a->E;
  KMOE_REQUIRE(a->K <= Eg && a->K <= 64 && a->E <= 1024 && Eg <= 1024, KMOE_ERR_SHAPE,
               "moe_forward: K=%d E=%d E_global=%d out of range", a->K, a->E, Eg);
  KMOE_REQUIRE(a->first_expert >= 0 && a->first_expert + a->E <= Eg, KMOE_ERR_SHAPE,
               "moe_forward: experts [%d, %d) are not among the %d the routing runs over", a->first_expert,
               a->first_expert + a->E, Eg);
  KMOE_REQUIRE(a->I_shared >= 0 && a->I_shared % mult == 0, KMOE_ERR_SHAPE,
               "moe_forward: I_shared=%d must be a non-negative multiple of %d", a->I_shared, mult);
  KMOE_REQUIRE(static_cast<long long>(a->M) * a->K <= (1 << 24), KMOE_ERR_SHAPE, "moe_forward: M*K too large");
  KMOE_REQUIRE(a->act_dtype == KMOE_DT_BF16 || a->act_dtype == KMOE_DT_F16, KMOE_ERR_UNSUPPORTED,
               "moe_forward: act_dtype=%d unknown", a->act_dtype);
  KMOE_REQUIRE(a->act_dtype == KMOE_DT_BF16 || a->format != KMOE_FMT_BF16 ||
                   (!a->w13_bias && !a->w2_bias && a->activation != KMOE_ACT_SWIGLUOAI),
               KMOE_ERR_UNSUPPORTED, "moe_forward: expert biases and swigluoai are built for bf16 only");
  // elements in 64 bytes of a weight row
  const int row64 = a->format == KMOE_FMT_BF16 ? 32 : (a->format == KMOE_FMT_W4A16 ? 128 : 64);
  KMOE_REQUIRE(a->w_layout == KMOE_W_ROWMAJOR ||
                   (a->w_layout == KMOE_W_TILED && a->H % row64 == 0 && a->I % row64 == 0),
               KMOE_ERR_SHAPE, "moe_forward: w_layout=%d needs H, I multiples of %d", a->w_layout, row64);
  KMOE_REQUIRE(a->I_shared == 0 || a->ws_layout == KMOE_W_ROWMAJOR ||
                   (a->ws_layout == KMOE_W_TILED && a->H % row64 == 0 && a->I_shared % row64 == 0),
               KMOE_ERR_SHAPE, "moe_forward: ws_layout=%d needs H, I_shared multiples of %d", a->ws_layout, row64);
  return KMOE_OK;
}

// The weight-streaming decode path (chunk-major codes, no row tiles) against the persistent tile kernel:
// the stream kernels re-read the weights once per 16-64 rows of an expert, so their time grows with the rows
// per expert; the tile kernel's hardly does. Measured cross-over with 64-row tiles: 10-12 rows per expert on
// both the Qwen3 and the DeepSeek-V3 shape.
// Pairs this launch expects to land on its own experts: all of them, or the share of an expert-parallel rank under
// uniform routing (the kernels are chosen by the rows per expert; any choice is correct for any routing).
long long local_pairs(const kmoe_moe_args* a) {
  const long long P = static_cast<long long>(a->M) * a->K;
  return a->E_global > a->E ? (P * a->E + a->E_global - 1) / a->E_global : P;
}

// KMOE_SORT_IN_GEMM=0 (read once) keeps the sort a launch of its own on the weight-streaming path too.
bool scan_allowed() {
  static const bool on = [] {
    const char* v = getenv("KMOE_SORT_IN_GEMM");
    return !(v && v[0] == '0');
  }();
  return on;
}

// KMOE_QUANT_IN_GEMM=0 (read once) keeps both quantisations launches of their own there.
bool quant_in_gemm_allowed() {
  static const bool on = [] {
    const char* v = getenv("KMOE_QUANT_IN_GEMM");
    return !(v && v[0] == '0');
  }();
  return on;
}

bool use_stream_path(const kmoe_moe_args* a) {
  const long long P = local_pairs(a);
  // a row-major shared expert cannot read the chunk-major codes this path quantises x into
  return a->format == KMOE_FMT_INT8 && a->w_layout == KMOE_W_TILED && (P + a->E - 1) / a->E <= 10 && a->M <= 1024 &&
         (a->I_shared == 0 || a->ws_layout == KMOE_W_TILED);
}

// Whether the routed gate_up GEMM runs on the weight-streaming kernel (and, 4-bit weights with long rows aside, the
// down GEMM as well).
bool routed_streams(const kmoe_moe_args* a) {
  if (a->w_layout != KMOE_W_TILED) return false;
  const long long rows = local_pairs(a);
  switch (a->format) {
    case KMOE_FMT_INT8: return use_stream_path(a);
    case KMOE_FMT_FP8_BLOCK: return streams_fp8(static_cast<int>(rows), a->E, a->H) && streams_fp8(static_cast<int>(rows), a->E, a->I);
    case KMOE_FMT_BF16:
      return streams_bf16(static_cast<int>(rows), a->E, a->H) && streams_bf16(static_cast<int>(rows), a->E, a->I) &&
             !a->w13_bias && !a->w2_bias && a->activation != KMOE_ACT_SWIGLUOAI;
    default:
      return w4_gate_up_streams(a->M * a->K, a->E_global > a->E ? static_cast<int>(rows) : 0, a->M, a->E, 2 * a->I, a->H) &&
             w4_rows_fit_32(a->M, a->H, a->H) && w4_rows_fit_32(static_cast<long long>(a->M) * a->K, a->I, a->I);
  }
}

// Whether this call may use the side stream: KMOE_FLAG_SIDE_STREAM of the call, unless the environment variable
// KMOE_SIDE_STREAM (read once) says 0 (never) or 1 (always).
bool wants_side_stream(const kmoe_moe_args* a) {
  static const int forced = [] {
    const char* v = getenv("KMOE_SIDE_STREAM");
    return (v && v[0]) ? (v[0] != '0' ? 1 : 0) : -1;
  }();
  return forced >= 0 ? forced == 1 : (a->flags & KMOE_FLAG_SIDE_STREAM) != 0;
}

// A shared expert of the routed experts' width runs inside the routed GEMM launches
// as one more ("tail") expert over rows [P, P+M): no extra launches, and its few
// workgroups overlap the routed experts' instead of leaving most CUs idle.
// fp8 on the weight-streaming kernel: the tail's 16-row slices read the shared weights once each, the pass of its own
// reads them once and costs its launches, unless a side stream hides them. DeepSeek-V3 dims, layer, us, folded / own
// pass: 23 tokens 949 / 1010, 128 1830 / 1873, 256 1942 / 1951, 288 1979 / 1974, 320 2035 / 2024; own pass on the side
// stream: 23 tokens 959, 64 1559 (folded 1557), 96 1748 (1754), 128 1822, 256 1895, 320 1983.
bool fold_shared(const kmoe_moe_args* a) {
  if (a->I_shared <= 0 || a->I_shared != a->I || a->ws_layout != a->w_layout) return false;
  if (a->format == KMOE_FMT_INT8) return true;
  if (a->format != KMOE_FMT_FP8_BLOCK || a->w_layout != KMOE_W_TILED || a->H > 8192 || a->I > 8192) return false;
  return !routed_streams(a) || a->M <= (wants_side_stream(a) ? 64 : 256);
}

// Whether the layer of a few tokens ends in one launch (few_down). It saves a launch or two, 4 to 8 us, and reads the down
// projection of an expert once per TOKEN that chose it (and of a shared expert that rides along once per token): what is read
// twice comes from the caches, and in the formats that are unpacked or scaled in the launch every reading is worked on again.
// Two bounds, both on what is read again. Under uniform routing, at about 6 MB a microsecond; layer, launches apart / in one, us, and
// those MB:
//   Qwen3 dims int8 1 token 23.7 / 18.9 (0), 4 42.5 / 36.6 (4), 8 60.4 / 56.6 (20), 10 64.9 / 62.2 (30), 12 74.4 / 74.0 (43);
//   bf16 1 token 26.3 / 22.3, 8 89.9 / 88.3 (39), 12 116 / 118 (85); 4-bit 1 token 21.4 / 18.6, 6 39.4 / 35.4 (6);
//   DeepSeek-V3 dims int8 1 token 95.3 / 87.5, 3 193.7 / 198.3 (40); fp8 1 token 95.3 / 88.6, 2 149 / 153 (18);
//   Kimi-K2 dims 4-bit 1 token 59.6 / 57.4, 3 116.9 / 116.0 (2).
// And with every token on the same experts (samples of one prompt), where the launch must not lose more than it gains under uniform
// routing. There one token's weights come from the L2 of the XCD that read them for the token before (column blocks keep their XCD)
// while an eighth of them fits its 4 MB, and from the memory-side cache beyond. Layer, us, apart / in one, uniform; same experts, and the MB:
//   Qwen3 dims int8 10 tokens 65.4 / 61.5; 27.2 / 26.2 (113), bf16 7 84.6 / 81.8; 26.9 / 27.0 (151), 4-bit 6 40.6 / 37.0; 20.7 / 22.0 (31),
//   8 44.0 / 40.5; 24.6 / 26.6 (44; left apart, as 7 are: samples of one prompt would pay 8 %), 128 experts of [4096 x 1536], 4-bit 3 59.4 / 56.7; 30.8 / 33.7 (50),
//   160 of [5120 x 1536], top 6, 3 58.1 / 57.0; 35.9 / 40.6 (47);
//   128 experts of [3072 x 4096], int8 2 tokens 60.5 / 53.8; 40.8 / 36.0 (50), 3 82.3 / 76.8; 42.4 / 45.9 (101), bf16 2 102.6 / 99.4; 57.5 / 61.9
//   (101), 4-bit 2 45.5 / 43.3; 29.9 / 31.0 (25), 3 62.8 / 60.9; 32.4 / 36.6 (50), fp8, 4 experts per token, 4 57.3 / 54.1; 29.3 / 28.2 (75);
//   DeepSeek-V3 dims int8 2 tokens 125.4 / 125.1; 87.4 / 104.3 (132); Kimi-K2 dims 4-bit 2 82.7 / 82.0; 56.7 / 62.7 (59).
bool few_down_pays(const kmoe_moe_args* a, bool fold) {
  if (a->I > kFewMaxI || a->K + (fold ? 1 : 0) > kFewMaxWaves) return false;
  // (what the GEMM launches refuse stays theirs to refuse)
  for (const void* t : {static_cast<const void*>(a->w2), static_cast<const void*>(a->w2_max), static_cast<const void*>(a->w2_scale),
                        static_cast<const void*>(a->ws2), static_cast<const void*>(a->ws2_max)})
    if (reinterpret_cast<uintptr_t>(t) & 15) return false;
  const double pairs = static_cast<double>(a->M) * a->K;
  double hit = a->E;
  for (int m = 0; m < a->M; ++m) hit *= 1.0 - static_cast<double>(a->K) / a->E;
  const double again = pairs - (a->E - hit) + (fold ? a->M - 1 : 0);
  const double bytes = static_cast<double>(a->H) * a->I * (a->format == KMOE_FMT_BF16 ? 2.0 : (a->format == KMOE_FMT_W4A16 ? 0.5 : 1.0));
  const double token = (a->K + (fold ? 1 : 0)) * bytes;
  const double same = (a->M - 1) * token;
  switch (a->format) {
    case KMOE_FMT_W4A16: return again * bytes <= 6e6 && same <= 42e6;
    case KMOE_FMT_FP8_BLOCK: return again * bytes <= 6e6 && same <= 80e6;
    default: return again * bytes <= 32e6 && same <= (token <= 8 * (4u << 20) ? 160e6 : 110e6);
  }
}

// Whether such a layer also begins in one launch (few_gate_up): up to kFewRouted tokens, so that routing is a wave each,
// whose rows leave room for five workgroups in a CU's LDS - fewer, and the launch no longer fills the chip at once (Kimi-K2
// dims, 4-bit, 1 token 57.1 -> 52.6 us, 2 tokens, three workgroups, 92.7 -> 98.9). Layer, us, apart / in one launch: Qwen3 dims int8 1
// token 16.8 / 13.3, 2 21.2 / 19.9, 4 32.6 / 29.6, bf16 1 20.3 / 18.8, 4 50.2 / 47.8, 4-bit 1 17.7 / 13.4, 4 26.0 / 24.7; DeepSeek-V3 dims int8 1 76.3 /
// 67.2, 2 135.2 / 130.2, 3 174.3 / 177.8, with the gate 1 86.4 / 75.6, fp8 1 80.1 / 71.5, 3 172.5 / 174.1; Kimi-K2 dims 4-bit 1 52.6 / 48.5.
bool few_gate_up_takes(const kmoe_moe_args* a) {
  if (a->M > kFewRouted || a->M * a->K > kWave || a->E > 8 * kWave || a->H > kFewRowBytes) return false;
  if (a->M * few_row_pitch(a->H, bf16_activations(a->format) ? 2 : 1, a->format == KMOE_FMT_FP8_BLOCK) > kFewRowBytes) return false;
  for (const void* t : {static_cast<const void*>(a->x), static_cast<const void*>(a->w13), static_cast<const void*>(a->w13_max),
                        static_cast<const void*>(a->w13_scale), static_cast<const void*>(a->ws13), static_cast<const void*>(a->ws13_max)})
    if (reinterpret_cast<uintptr_t>(t) & 15) return false;
  return true;
}

// What a layer whose gate_up launch routes its tokens itself hands to it.
struct FewRouted {
  RouteArgs route;
  bool sigmoid;
  const uint16_t* x;
};

// One expert-MLP pass (gate_up + SiLU-mul, requantise, down) over `rows` rows in
// the layer's format. `x_rows` is what the first GEMM reads: quantised codes, or
// the bf16 activations themselves for KMOE_FMT_BF16.
struct MlpPass {
  int format;
  const void* x_rows;      // [*, H]
  const float* x_aux;      // row maxes / group scales (NULL for bf16)
  const int32_t* row_src;  // gather for the first GEMM (NULL: identity)
  int src_div;
  const void *w13, *w2;
  const float *w13_aux, *w2_aux;
  const int32_t* lod;
  int E, H, I, rows;
  int rows_hint;   // 0, or the rows expected to be live (an expert-parallel share): see kmoe_gemm_*_args
  uint16_t* act;   // [rows, I] bf16
  void* actq;      // [rows, I] codes
  float* act_aux;  // [rows] or [rows, I/128]
  uint16_t* out;   // [rows, H] bf16
  int w_layout;    // KMOE_W_*
  bool stream;     // INT8 + tiled weights: chunk-major codes and the weight-streaming GEMM
  int x_count;     // rows of x_rows (chunk-major addressing)
  // INT8, FP8 tail expert (folded shared expert): rows [rows, rows + tail_rows) of act/actq/out
  const void *w13_tail, *w2_tail;
  const float *w13_aux_tail, *w2_aux_tail;
  int tail_rows;
  // BF16 expert-bias branch
  const uint16_t *w13_bias, *w2_bias;
  int oai;  // 1: gate_up rows interleaved, gpt-oss activation
  float act_alpha, act_limit;
  // W4A16: group scales of the packed weights
  const uint16_t *w13_scale, *w2_scale;
  int group_size, scale_layout;
  int variant;  // INT8: kernel variant of the two GEMMs (0: from the shape)
  int act_dtype;  // INT8, BF16: KMOE_DT_* of x_rows' source, act and out (BF16: of the weights too)
  // weight-streaming path: the gate_up launch sorts the routed pairs itself (row_src is then NULL and lod is
  // what that launch writes); slots: the down launch has a column of workgroups per pair, as the gate_up launch had
  const StreamScan* scan;
  const StreamSlots* slots;
  bool quant_in_gemm;  // the down launch quantises its rows itself: no launch between the two GEMMs
  const FewRouted* first;  // a few tokens: the gate_up launch routes, quantises and sorts (scan: where it leaves the sort)
  bool few_down;       // a few tokens: one launch for quantisation, down projection and combine ends the layer
};

int run_gemm(const MlpPass& m, bool first, kmoe_stream_t stream) {
  const int n = first ? 2 * m.I : m.H;
  const int k = first ? m.H : m.I;
  const void* a = first ? m.x_rows : (bf16_activations(m.format) ? static_cast<const void*>(m.act) : m.actq);
  const float* a_aux = first ? m.x_aux : m.act_aux;
  const void* w = first ? m.w13 : m.w2;
  const float* w_aux = first ? m.w13_aux : m.w2_aux;
  uint16_t* y = first ? m.act : m.out;
  const int64_t ldy = first ? m.I : m.H;
  const int act = first ? KMOE_ACT_SWIGLU : KMOE_ACT_NONE;
  const int32_t* row_src = first ? m.row_src : nullptr;
  const int src_div = first ? m.src_div : 1;
  if (m.format == KMOE_FMT_INT8) {
    kmoe_gemm_i8_args g = {};
    g.a = static_cast<const int8_t*>(a);
    g.lda = k;
    g.a_max = a_aux;
    g.row_src = row_src;
    g.src_div = src_div;
    g.w = static_cast<const int8_t*>(w);
    g.w_max = w_aux;
    g.lod = m.lod;
    g.E = m.E;
    g.n = n;
    g.k = k;
    g.rows = m.rows;
    g.rows_hint = m.rows_hint;
    g.y = y;
    g.ldy = ldy;
    g.act = act;
    g.w_layout = m.w_layout;
    g.variant = m.variant;
    g.act_dtype = m.act_dtype;
    if (m.stream) {
      g.a_layout = KMOE_A_CHUNKED;
      g.a_rows = first ? m.x_count : m.rows + m.tail_rows;
    }
    if (m.tail_rows > 0) {
      g.w_tail = static_cast<const int8_t*>(first ? m.w13_tail : m.w2_tail);
      g.w_max_tail = first ? m.w13_aux_tail : m.w2_aux_tail;
      g.tail_row0 = m.rows;
      g.tail_rows = m.tail_rows;
      g.tail_src0 = first ? 0 : m.rows;  // gate_up reads token rows, down reads its own act rows
    }
    const StreamQuant quant{m.act, m.I, static_cast<int8_t*>(m.actq), m.act_aux};
    return grouped_gemm_i8_checked(&g, stream, first ? m.scan : nullptr, !first && m.quant_in_gemm ? &quant : nullptr,
                                   first ? nullptr : m.slots);
  }
  if (m.format == KMOE_FMT_FP8_BLOCK) {
    kmoe_gemm_fp8_args g = {};
    g.a = static_cast<const uint8_t*>(a);
    g.lda = k;
    g.a_scale = a_aux;
    g.row_src = row_src;
    g.src_div = src_div;
    g.w = static_cast<const uint8_t*>(w);
    g.w_scale = w_aux;
    g.act_dtype = m.act_dtype;
    g.lod = m.lod;
    g.E = m.E;
    g.n = n;
    g.k = k;
    g.rows = m.rows;
    g.rows_hint = m.rows_hint;
    g.y = y;
    g.ldy = ldy;
    g.act = act;
    g.w_layout = m.w_layout;
    g.variant = m.variant;
    if (m.tail_rows > 0) {
      g.w_tail = static_cast<const uint8_t*>(first ? m.w13_tail : m.w2_tail);
      g.w_scale_tail = first ? m.w13_aux_tail : m.w2_aux_tail;
      g.tail_row0 = m.rows;
      g.tail_rows = m.tail_rows;
      g.tail_src0 = first ? 0 : m.rows;  // gate_up reads token rows, down reads its own act rows
    }
    return grouped_gemm_fp8_checked(&g, stream, first ? m.scan : nullptr, first ? nullptr : m.slots);
  }
  if (m.format == KMOE_FMT_W4A16) {
    kmoe_gemm_w4_args g = {};
    g.a = static_cast<const uint16_t*>(a);
    g.lda = k;
    g.row_src = row_src;
    g.src_div = src_div;
    g.w = static_cast<const uint8_t*>(w);
    g.w_scale = first ? m.w13_scale : m.w2_scale;
    g.group_size = m.group_size;
    g.scale_layout = m.scale_layout;
    g.lod = m.lod;
    g.E = m.E;
    g.n = n;
    g.k = k;
    g.rows = m.rows;
    g.rows_hint = m.rows_hint;
    g.y = y;
    g.ldy = ldy;
    g.act = act;
    g.w_layout = m.w_layout;
    g.act_dtype = m.act_dtype;
    return grouped_gemm_w4a16_checked(&g, stream, first ? m.scan : nullptr, first ? nullptr : m.slots,
                                      first ? m.x_count : m.rows);
  }
  kmoe_gemm_bf16_args g = {};
  g.a = static_cast<const uint16_t*>(a);
  g.lda = k;
  g.row_src = row_src;
  g.src_div = src_div;
  g.w = static_cast<const uint16_t*>(w);
  g.lod = m.lod;
  g.E = m.E;
  g.n = n;
  g.k = k;
  g.rows = m.rows;
  g.rows_hint = m.rows_hint;
  g.y = y;
  g.ldy = ldy;
  g.act = first && m.oai ? KMOE_ACT_SWIGLUOAI : act;
  g.w_layout = m.w_layout;
  g.bias = first ? m.w13_bias : m.w2_bias;
  g.act_alpha = m.act_alpha;
  g.act_limit = m.act_limit;
  g.act_dtype = m.act_dtype;
  return grouped_gemm_bf16_checked(&g, stream, first ? m.scan : nullptr, first ? nullptr : m.slots);
}

// Group scales of packed 4-bit weights, as the decode kernels address them.
template <class P>
void set_group_scales(P* p, const uint16_t* scale, int k, int group_size, int layout) {
  const bool frag16 = layout == KMOE_S_FRAG16;
  p->w_scale = scale;
  p->groups = k / group_size;
  p->s_ch = frag16 ? 1 : p->groups;
  p->s_g = frag16 ? 16 : 1;
  p->gs32 = group_size / 32;
  p->gs_shift = (p->gs32 & (p->gs32 - 1)) == 0 ? __builtin_ctz(p->gs32) : -1;
}

// The launch of a few tokens' down projection, combine included; gate_up has left its rows in m.act.
int run_few_down(const MlpPass& m, const kmoe_moe_args* a, const int32_t* ids, const int32_t* moe_index, const float* topk_w, hipStream_t stream) {
  FewDown p = {};
  p.M = a->M;
  p.K = a->K;
  p.H = m.H;
  p.I = m.I;
  p.kbytes = m.format == KMOE_FMT_BF16 ? 2 * m.I : (m.format == KMOE_FMT_W4A16 ? m.I / 2 : m.I);
  p.ids = ids;
  p.moe_index = moe_index;
  p.topk_w = topk_w;
  p.act = m.act;
  p.rows = m.rows + m.tail_rows;
  p.codes = static_cast<int8_t*>(m.actq);
  p.code_aux = m.act_aux;
  p.w = static_cast<const int8_t*>(m.w2);
  p.w_aux = m.w2_aux;
  if (m.tail_rows > 0) {
    p.w_tail = static_cast<const int8_t*>(m.w2_tail);
    p.w_aux_tail = m.w2_aux_tail;
  }
  if (m.format == KMOE_FMT_W4A16) set_group_scales(&p, m.w2_scale, m.I, m.group_size, m.scale_layout);
  p.down = m.out;
  p.out_scale = a->out_scale;
  p.shared_scale = a->shared_scale == 0.0f ? 1.0f : a->shared_scale;
  p.out = a->out;
  p.f16 = m.act_dtype == KMOE_DT_F16;
  return few_down(p, m.format, stream);
}

// The launch that routes up to kFewRouted tokens and runs their gate_up projection.
int run_few_gate_up(const MlpPass& m, hipStream_t stream) {
  FewGateUp p = {};
  p.route = m.first->route;
  p.H = m.H;
  p.I = m.I;
  p.kbytes = m.format == KMOE_FMT_BF16 ? 2 * m.H : (m.format == KMOE_FMT_W4A16 ? m.H / 2 : m.H);
  p.x = m.first->x;
  p.w = static_cast<const int8_t*>(m.w13);
  p.w_aux = m.w13_aux;
  if (m.tail_rows > 0) {
    p.w_tail = static_cast<const int8_t*>(m.w13_tail);
    p.w_aux_tail = m.w13_aux_tail;
  }
  if (m.format == KMOE_FMT_W4A16) set_group_scales(&p, m.w13_scale, m.H, m.group_size, m.scale_layout);
  p.sort = *m.scan;
  p.act = m.act;
  p.f16 = m.act_dtype == KMOE_DT_F16;
  return few_gate_up(p, m.format, m.first->sigmoid, stream);
}

template <class Mark>
int run_mlp(const MlpPass& m, kmoe_stream_t stream, Mark&& mark) {
  int rc;
  const char* whose = m.row_src || m.scan ? "routed experts" : "shared expert";
  mark(KMOE_STAGE_GEMM1, 0);
  if (tracing_kernels()) note_kernel("[gate_up, %s]", whose);
  rc = m.first ? run_few_gate_up(m, as_stream(stream)) : run_gemm(m, true, stream);
  if (rc) return rc;
  mark(KMOE_STAGE_GEMM1, 1);
  mark(KMOE_STAGE_QUANT2, 0);
  if (m.few_down) {  // (the rest is the caller's)
    mark(KMOE_STAGE_QUANT2, 1);
    return KMOE_OK;
  }
  if (m.format == KMOE_FMT_INT8 && m.quant_in_gemm) {
    // (the down launch does it)
  } else if (m.format == KMOE_FMT_INT8) {
    const int qrows = m.rows + m.tail_rows;
    rc = m.stream ? kmoe_quant_i8_rows_chunked_dt(m.act, m.I, qrows, m.I, static_cast<int8_t*>(m.actq), m.act_aux,
                                                  m.act_dtype, stream)
                  : kmoe_quant_i8_rows_dt(m.act, m.I, qrows, m.I, static_cast<int8_t*>(m.actq), m.I, m.act_aux,
                                          m.act_dtype, stream);
  } else if (m.format == KMOE_FMT_FP8_BLOCK) {
    rc = kmoe_quant_fp8_group128_dt(m.act, m.I, m.rows + m.tail_rows, m.I, static_cast<uint8_t*>(m.actq), m.I, m.act_aux,
                                    m.act_dtype, stream);
  }
  if (rc) return rc;
  mark(KMOE_STAGE_QUANT2, 1);
  mark(KMOE_STAGE_GEMM2, 0);
  if (tracing_kernels()) note_kernel("[down, %s]", whose);
  rc = run_gemm(m, false, stream);
  if (rc) return rc;
  mark(KMOE_STAGE_GEMM2, 1);
  return KMOE_OK;
}

}  // namespace

extern "C" int kmoe_moe_workspace_layout(const kmoe_moe_args* a, kmoe_moe_layout* L) {
  if (int rc = check_shape(a)) return rc;
  KMOE_REQUIRE(L, KMOE_ERR_NULL, "moe_workspace_layout: layout is NULL");
  const size_t M = a->M, H = a->H, E = a->E, K = a->K, I = a->I, P = M * K, Is = a->I_shared;
  const bool quant = !bf16_activations(a->format);
  const bool fp8 = a->format == KMOE_FMT_FP8_BLOCK;
  const bool fold = fold_shared(a);
  const size_t R = P + (fold ? M : 0);  // rows of the routed intermediates (+ folded shared expert rows)
  const size_t Ms = fold ? 0 : (Is ? M : 0);  // rows of the separate shared-expert intermediates
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align_up(bytes ? bytes : 1, 256);
    return at;
  };
  L->topk_w = take(P * 4);
  L->topk_ids = take(P * 4);
  L->moe_index = take(P * 4);
  L->sorted_src = take(P * 4);
  L->expert_m = take(E * 4);
  L->lod = take((E + 1) * 4);
  // (launches with a column of workgroups per pair keep their row ranges where the sort's launch would have its own)
  L->align_ws = take(std::max(kmoe_align_workspace_bytes(static_cast<int>(P), a->E), P <= kStreamSlotMaxPairs ? P * sizeof(int2) : 0));
  L->xq = take(quant ? M * H : 0);
  L->xmax = take(quant ? M * 4 * (fp8 ? H / 128 : 1) : 0);
  L->act = take(R * I * 2);
  L->actq = take(quant ? R * I : 0);
  L->actmax = take(quant ? R * 4 * (fp8 ? I / 128 : 1) : 0);
  L->down = take(R * H * 2);
  L->sh_lod = take(2 * 4);
  L->sh_act = take(Ms * Is * 2);
  L->sh_actq = take(quant ? Ms * Is : 0);
  L->sh_actmax = take(quant ? Ms * 4 * (fp8 ? Is / 128 : 1) : 0);
  L->sh_out = take(Ms * H * 2);
  int ks = 0, mf = 0;
  if (a->w_gate && a->H % 32 == 0) router_plan(a->M, a->H, a->E_global > 0 ? a->E_global : a->E, &ks, &mf);
  L->n_logit_planes = ks;
  L->logit_planes = take(ks ? static_cast<size_t>(ks) * M * (a->E_global > 0 ? a->E_global : E) * 4 : 0);
  L->total_bytes = off;
  L->codes_chunked = use_stream_path(a) ? 1 : 0;
  return KMOE_OK;
}

namespace {

// A shared expert that does not ride in the routed launches (another width; larger fp8 decode batches) is a chain of
// small launches that depends on the layer's input only. It runs on a stream of the library's own, forked from
// the caller's stream after the first quantisation and joined back before the combine, so that it hides under
// the routed GEMMs instead of adding its launches' latencies to the layer (DeepSeek-V3 fp8, 256 tokens: 56 us of
// 1.95 ms). Only for calls that ask for it (KMOE_FLAG_SIDE_STREAM): by default every launch goes to the caller's
// stream. One stream and two events per GPU, created on the first call that wants them and is not being
// captured (default priority, non-blocking); work of consecutive calls is ordered on it like on any stream.
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  bool failed = false;
};
constexpr int kSideDevices = 64;
SideStream g_side[kSideDevices];
std::mutex g_side_mutex;

// The side stream of the current device, or NULL: not created yet while the caller's stream is being captured (a
// capture must not be the first to ask), or the runtime refused.
SideStream* side_stream(hipStream_t main) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kSideDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_side_mutex);
  SideStream& sd = g_side[dev];
  if (sd.stream) return &sd;
  if (sd.failed) return nullptr;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(main, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (hipStreamCreateWithFlags(&sd.stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&sd.fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&sd.join, hipEventDisableTiming) != hipSuccess) {
    (void)hipGetLastError();
    sd.failed = true;
    sd.stream = nullptr;
    return nullptr;
  }
  return &sd;
}

int moe_forward_impl(const kmoe_moe_args* a, void* workspace, size_t workspace_bytes, kmoe_stream_t stream,
                     bool may_fork);
void learn_static_workspace(hipStream_t stream);

}  // namespace

extern "C" int kmoe_moe_forward(const kmoe_moe_args* a, void* workspace, size_t workspace_bytes,
                                kmoe_stream_t stream) {
  learn_static_workspace(as_stream(stream));  // (so that a later captured kmoe_moe_forward_static finds the address)
  return moe_forward_impl(a, workspace, workspace_bytes, stream, true);
}

namespace {

int moe_forward_impl(const kmoe_moe_args* a, void* workspace, size_t workspace_bytes, kmoe_stream_t stream,
                     bool may_fork) {
  kmoe_moe_layout L;
  if (int rc = kmoe_moe_workspace_layout(a, &L)) return rc;
  if (a->M == 0) return KMOE_OK;
  const bool quant = !bf16_activations(a->format);
  KMOE_REQUIRE((a->logits || a->w_gate) && a->x && a->w13 && a->w2 && a->out, KMOE_ERR_NULL,
               "moe_forward: NULL tensor pointer");
  KMOE_REQUIRE(a->logits || (a->H % 32 == 0 && (reinterpret_cast<uintptr_t>(a->w_gate) & 15) == 0 &&
                             (reinterpret_cast<uintptr_t>(a->x) & 15) == 0),
               KMOE_ERR_SHAPE, "moe_forward: the router GEMM needs H %% 32 == 0 and 16-byte aligned x, w_gate");
  KMOE_REQUIRE(!quant || (a->w13_max && a->w2_max), KMOE_ERR_NULL, "moe_forward: weight max/scale pointers are NULL");
  KMOE_REQUIRE(a->format != KMOE_FMT_W4A16 || (a->w13_scale && a->w2_scale), KMOE_ERR_NULL,
               "moe_forward: group scale pointers are NULL");
  KMOE_REQUIRE(a->I_shared == 0 || (a->ws13 && a->ws2 && (!quant || (a->ws13_max && a->ws2_max))), KMOE_ERR_NULL,
               "moe_forward: shared expert pointers are NULL");
  KMOE_REQUIRE(a->scoring == KMOE_SCORE_SOFTMAX || a->scoring == KMOE_SCORE_SIGMOID, KMOE_ERR_UNSUPPORTED,
               "moe_forward: scoring=%d unknown", a->scoring);
  KMOE_REQUIRE(a->activation == 0 || a->activation == KMOE_ACT_SWIGLU ||
                   (a->activation == KMOE_ACT_SWIGLUOAI && a->format == KMOE_FMT_BF16),
               KMOE_ERR_UNSUPPORTED, "moe_forward: activation=%d (swigluoai goes with bf16 weights only)", a->activation);
  KMOE_REQUIRE((!a->w13_bias && !a->w2_bias) || a->format == KMOE_FMT_BF16, KMOE_ERR_UNSUPPORTED,
               "moe_forward: expert biases go with bf16 weights only");
  KMOE_REQUIRE(!a->w13_bias || a->activation == KMOE_ACT_SWIGLUOAI, KMOE_ERR_UNSUPPORTED,
               "moe_forward: a gate_up bias goes with the swigluoai activation");
  KMOE_REQUIRE(workspace, KMOE_ERR_WORKSPACE, "moe_forward: workspace is NULL (need %zu bytes)", L.total_bytes);
  KMOE_REQUIRE(workspace_bytes >= L.total_bytes, KMOE_ERR_WORKSPACE, "moe_forward: workspace %zu < %zu bytes",
               workspace_bytes, L.total_bytes);
  KMOE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, KMOE_ERR_WORKSPACE,
               "moe_forward: workspace must be 256-byte aligned");

  char* ws = static_cast<char*>(workspace);
  auto at = [&](size_t off) { return static_cast<void*>(ws + off); };
  float* topk_w = static_cast<float*>(at(L.topk_w));
  int32_t* topk_ids = static_cast<int32_t*>(at(L.topk_ids));
  int32_t* moe_index = static_cast<int32_t*>(at(L.moe_index));
  int32_t* sorted_src = static_cast<int32_t*>(at(L.sorted_src));
  int32_t* lod = static_cast<int32_t*>(at(L.lod));
  const int M = a->M, H = a->H, E = a->E, K = a->K, I = a->I, P = M * K;
  const int Eg = a->E_global > 0 ? a->E_global : E;  // experts the routing runs over (an expert-parallel share: more than E)
  int rc = KMOE_OK;
  auto mark = [&](int stage, int end) {
    if (!a->stage_events) return;
    void* ev = a->stage_events[2 * stage + end];
    if (ev) (void)hipEventRecord(static_cast<hipEvent_t>(ev), as_stream(stream));
  };

  // 0. router logits if the caller handed over the gate weight instead: split-K partial planes,
  //    which the routing kernel adds up as it loads them (timed as part of the routing stage)
  const bool stream_mode = use_stream_path(a);
  bool quant_done = false;
  mark(KMOE_STAGE_ROUTING, 0);
  const bool f16 = a->act_dtype == KMOE_DT_F16;
  LogitsView logits{a->logits, 1, 0, (a->flags & KMOE_FLAG_LOGITS_ACT_DTYPE) ? (f16 ? 2 : 1) : 0};
  if (!a->logits) {
    int mf = 0, planes = 1;
    router_plan(M, H, Eg, &planes, &mf);
    float* buf = static_cast<float*>(at(L.logit_planes));
    logits = LogitsView{buf, planes, static_cast<size_t>(M) * Eg, 0};
    rc = router_gemm_planes(a->x, H, a->w_gate, M, H, Eg, buf, logits.plane_stride, Eg, planes, mf, as_stream(stream), f16);
    if (rc) return rc;
  }
  // 1. routing; for the quantised formats together with step 3 (independent work, one launch)
  const bool scan_in_gemm = routed_streams(a) && Eg == E && a->first_expert == 0 && P <= kStreamScanMaxPairs &&
                            M <= kStreamScanMaxRows && scan_allowed();
  // Fewer pairs than experts: a column of workgroups per pair instead of per expert.
  const bool per_pair = scan_in_gemm && P < E && P <= kStreamSlotMaxPairs;
  const bool fold = fold_shared(a);
  const bool few = per_pair && (a->I_shared == 0 || fold) && quant_in_gemm_allowed();
  const bool few_down = few && few_down_pays(a, fold);
  const bool few_routed = few && few_gate_up_takes(a);
  RouteArgs route{logits, a->bias, M, Eg, K, a->renormalize, a->n_group, a->topk_group, a->routed_scale, topk_w, topk_ids};
  if (few_routed)
    rc = check_route(&route, a->scoring == KMOE_SCORE_SIGMOID);  // (the gate_up launch does it, and steps 2 and 3)
  else
    rc = route_and_quantise(route, a->scoring == KMOE_SCORE_SIGMOID, a->format, a->x, H, at(L.xq),
                            static_cast<float*>(at(L.xmax)), stream_mode, f16, &quant_done, as_stream(stream));
  if (rc) return rc;
  mark(KMOE_STAGE_ROUTING, 1);
  // 2. stable sort of the routed pairs by expert. On the weight-streaming path (a few rows per expert) the gate_up
  // launch does it in its prologue and writes the same four arrays: one launch and its round trips less
  // (Qwen3 decode: 4.8 us of 125). Not for an expert-parallel share (pairs of other ranks' experts get no row).
  mark(KMOE_STAGE_ALIGN, 0);
  int2* slot_rows = per_pair ? static_cast<int2*>(at(L.align_ws)) : nullptr;
  const StreamScan scan{topk_ids, P, lod, static_cast<int32_t*>(at(L.expert_m)), moe_index, sorted_src, slot_rows};
  const StreamSlots slots{topk_ids, slot_rows, P};
  if (!scan_in_gemm) {
    rc = kmoe_align_local(topk_ids, P, E, a->first_expert, moe_index, sorted_src, static_cast<int32_t*>(at(L.expert_m)), lod,
                          at(L.align_ws), kmoe_align_workspace_bytes(P, E), stream);
    if (rc) return rc;
  }
  mark(KMOE_STAGE_ALIGN, 1);
  // 3. quantise each TOKEN row once (the reference quantises the K-times expanded copy; same values)
  mark(KMOE_STAGE_QUANT1, 0);
  const void* x_rows = a->x;
  if (quant_done) {
    x_rows = at(L.xq);
  } else if (few_routed) {
  } else if (a->format == KMOE_FMT_INT8) {
    rc = stream_mode ? kmoe_quant_i8_rows_chunked_dt(a->x, H, M, H, static_cast<int8_t*>(at(L.xq)),
                                                     static_cast<float*>(at(L.xmax)), a->act_dtype, stream)
                     : kmoe_quant_i8_rows_dt(a->x, H, M, H, static_cast<int8_t*>(at(L.xq)), H,
                                             static_cast<float*>(at(L.xmax)), a->act_dtype, stream);
    x_rows = at(L.xq);
  } else if (a->format == KMOE_FMT_FP8_BLOCK) {
    rc = kmoe_quant_fp8_group128_dt(a->x, H, M, H, static_cast<uint8_t*>(at(L.xq)), H, static_cast<float*>(at(L.xmax)),
                                    a->act_dtype, stream);
    x_rows = at(L.xq);
  }
  if (rc) return rc;
  mark(KMOE_STAGE_QUANT1, 1);

  // 4-6. routed experts: gate_up GEMM (+SiLU-mul, rows gathered through the sort), requantise, down GEMM
  MlpPass routed = {};
  routed.format = a->format;
  routed.x_rows = x_rows;
  routed.x_aux = quant ? static_cast<const float*>(at(L.xmax)) : nullptr;
  routed.row_src = scan_in_gemm ? nullptr : sorted_src;
  routed.scan = scan_in_gemm ? &scan : nullptr;
  routed.slots = per_pair ? &slots : nullptr;
  routed.src_div = K;
  routed.w13 = a->w13;
  routed.w2 = a->w2;
  routed.w13_aux = a->w13_max;
  routed.w2_aux = a->w2_max;
  routed.lod = lod;
  routed.E = E;
  routed.H = H;
  routed.I = I;
  routed.rows = P;
  routed.rows_hint = a->E_global > E ? static_cast<int>(local_pairs(a)) : 0;
  routed.act = static_cast<uint16_t*>(at(L.act));
  routed.actq = at(L.actq);
  routed.act_aux = static_cast<float*>(at(L.actmax));
  routed.out = static_cast<uint16_t*>(at(L.down));
  routed.w_layout = a->w_layout;
  routed.w13_scale = a->w13_scale;
  routed.w2_scale = a->w2_scale;
  routed.group_size = a->group_size;
  routed.scale_layout = a->w_scale_layout;
  routed.act_dtype = a->act_dtype;
  if (a->format == KMOE_FMT_BF16) {
    routed.w13_bias = a->w13_bias;
    routed.w2_bias = a->w2_bias;
    routed.oai = a->activation == KMOE_ACT_SWIGLUOAI;
    routed.act_alpha = a->act_alpha;
    routed.act_limit = a->act_limit;
  }
  routed.stream = stream_mode;
  // Down projections up to 1024 wide quantise their rows in the launch's prologue (Qwen3 decode: one 4.5 us launch
  // and its gap less); wider rows would not fit the workgroup's LDS copy next to three resident workgroups per CU.
  routed.quant_in_gemm = stream_mode && I <= kStreamQuantMaxK && quant_in_gemm_allowed();
  routed.x_count = M;
  uint32_t magic;
  const bool macro = a->tile_variant == 23 && macro_tile_takes(H, E, fold) && macro_tile_takes(I, E, fold) && macro_tile_divides(K, &magic);
  if (a->format == KMOE_FMT_INT8 && !stream_mode && a->w_layout == KMOE_W_TILED && a->tile_variant >= 5 &&
      (a->tile_variant <= 22 || macro) && (local_pairs(a) + E - 1) / E > 10 && H >= 128 && I >= 128)
    routed.variant = a->tile_variant;
  const int tv = a->tile_variant;
  if (a->format == KMOE_FMT_FP8_BLOCK && a->w_layout == KMOE_W_TILED && (local_pairs(a) + E - 1) / E > 10 &&
      (tv == 5 || tv == 6 || tv == 8 || (tv >= 11 && tv <= 14) || (tv >= 17 && tv <= 20) || macro))
    routed.variant = tv;
  if (fold) {
    routed.w13_tail = a->ws13;
    routed.w2_tail = a->ws2;
    routed.w13_aux_tail = a->ws13_max;
    routed.w2_aux_tail = a->ws2_max;
    routed.tail_rows = M;
  }
  const FewRouted first{route, a->scoring == KMOE_SCORE_SIGMOID, a->x};
  routed.first = few_routed ? &first : nullptr;
  routed.few_down = few_down;
  // 7. dense shared expert on all M rows: the grouped GEMM with a single expert whose lod is {0, M}. With a side
  // stream it is enqueued there BEFORE the routed pass (it reads x / its codes only) and joined after it.
  const uint16_t* shared_out = fold ? routed.out + static_cast<size_t>(P) * H : nullptr;
  const bool own_pass = a->I_shared > 0 && !fold;
  SideStream* side =
      own_pass && may_fork && !a->stage_events && wants_side_stream(a) ? side_stream(as_stream(stream)) : nullptr;
  auto shared_pass = [&](kmoe_stream_t st) -> int {
    int32_t* dense_lod = static_cast<int32_t*>(at(L.sh_lod));
    int rcs = fill_dense_lod(dense_lod, stream_mode ? 0 : M, as_stream(st));  // (streaming path: see below)
    if (rcs) return rcs;
    MlpPass sh = routed;
    // the expert-bias branch belongs to the routed experts only: a dense shared MLP has no per-expert
    // bias and uses the plain SiLU-mul over [gate | up] rows
    sh.w13_bias = nullptr;
    sh.w2_bias = nullptr;
    sh.oai = 0;
    sh.tail_rows = 0;
    sh.row_src = nullptr;
    sh.scan = nullptr;
    sh.slots = nullptr;
    sh.quant_in_gemm = false;
    sh.first = nullptr;
    sh.few_down = false;
    sh.src_div = 1;
    sh.w13 = a->ws13;
    sh.w2 = a->ws2;
    sh.w_layout = a->ws_layout;
    sh.w13_aux = a->ws13_max;
    sh.w2_aux = a->ws2_max;
    sh.lod = dense_lod;
    sh.E = 1;
    sh.I = a->I_shared;
    sh.rows = M;
    sh.rows_hint = 0;
    sh.variant = 0;  // (a tuning variant of the routed GEMMs does not apply to the dense pass)
    if (stream_mode) {
      // On the weight-streaming path a dense expert is best run as the launch's TAIL expert: the kernel cuts
      // a tail's rows into 16- or 32-row slices for as many workgroups, while one routed expert with M rows
      // is one column of workgroups that walks its rows in passes (measured at 64 tokens, hidden 2048:
      // the pass of a shared expert of intermediate size 1536 took 56 us, now 22; of size 6144, 97 -> 36 us).
      // The routed expert list is then one expert without rows.
      sh.rows = 0;
      sh.tail_rows = M;
      sh.w13_tail = a->ws13;
      sh.w2_tail = a->ws2;
      sh.w13_aux_tail = a->ws13_max;
      sh.w2_aux_tail = a->ws2_max;
      sh.variant = M <= 128 ? 1 : (M <= 256 ? 2 : 4);  // rows per slice: 16, 32, 64
    }
    sh.act = static_cast<uint16_t*>(at(L.sh_act));
    sh.actq = at(L.sh_actq);
    sh.act_aux = static_cast<float*>(at(L.sh_actmax));
    sh.out = static_cast<uint16_t*>(at(L.sh_out));
    rcs = run_mlp(sh, st, [](int, int) {});
    if (rcs) return rcs;
    shared_out = sh.out;
    return KMOE_OK;
  };
  if (side) {
    // (record and wait are one step under the lock: the events are shared by every caller on this GPU, and a
    // wait refers to the event's latest record)
    auto hand_over = [](hipEvent_t ev, hipStream_t from, hipStream_t to) {
      std::lock_guard<std::mutex> lock(g_side_mutex);
      hipError_t err = hipEventRecord(ev, from);
      if (err == hipSuccess) err = hipStreamWaitEvent(to, ev, 0);
      return err;
    };
    hipError_t e = hand_over(side->fork, as_stream(stream), side->stream);
    KMOE_REQUIRE(e == hipSuccess, KMOE_ERR_LAUNCH, "moe_forward: fork to the side stream: %s", hipGetErrorString(e));
    const int rc_side = shared_pass(side->stream);
    rc = rc_side ? rc_side : run_mlp(routed, stream, mark);
    // joined in any case, after the routed pass is in the caller's stream: a captured side stream must come back
    // to the stream it forked from
    e = hand_over(side->join, side->stream, as_stream(stream));
    if (rc) return rc;
    KMOE_REQUIRE(e == hipSuccess, KMOE_ERR_LAUNCH, "moe_forward: join of the side stream: %s", hipGetErrorString(e));
  } else {
    rc = run_mlp(routed, stream, mark);
    if (rc) return rc;
  }
  mark(KMOE_STAGE_SHARED, 0);
  if (own_pass && !side) {
    rc = shared_pass(stream);
    if (rc) return rc;
  }
  mark(KMOE_STAGE_SHARED, 1);
  if (routed.few_down) {  // 8. with the down projection
    mark(KMOE_STAGE_GEMM2, 0);
    if (tracing_kernels()) note_kernel("[down, routed experts]");
    rc = run_few_down(routed, a, topk_ids, moe_index, topk_w, as_stream(stream));
    mark(KMOE_STAGE_GEMM2, 1);
    mark(KMOE_STAGE_SHARED, 0);
    mark(KMOE_STAGE_SHARED, 1);
    mark(KMOE_STAGE_COMBINE, 0);
    mark(KMOE_STAGE_COMBINE, 1);
    return rc;
  }
  // 8. weighted combine (+ caller epilogue)
  mark(KMOE_STAGE_COMBINE, 0);
  // shared_scale == 0 (a zeroed field) means 1
  rc = kmoe_combine_dt(static_cast<uint16_t*>(at(L.down)), H, moe_index, topk_w, nullptr, M, K, H, a->out_scale,
                       shared_out, H, a->shared_scale == 0.0f ? 1.0f : a->shared_scale, a->out, H, a->act_dtype,
                       stream);
  mark(KMOE_STAGE_COMBINE, 1);
  return rc;
}

}  // namespace

// ---- the layer for callers that cannot hand over a workspace -------------------------------
// kmoe_moe_forward with its workspace in a file-scope device array. The array's name is only a
// host-side handle: its device address is asked for once per GPU (each GPU holds its own copy at
// its own address) and that address is what the kernels get.
static __device__ __align__(256) unsigned char scratch[KMOE_STATIC_WORKSPACE_BYTES];

namespace {

constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mutex;

// Device address of `scratch` on the current GPU. It is looked up once per GPU, by the first call whose stream is
// not being captured (the lookup is not a stream operation and may be what makes the runtime load the array); a
// captured call that finds it missing is refused.
int static_workspace(void** out, hipStream_t stream) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return fail(KMOE_ERR_LAUNCH, "moe_forward_static: hipGetDevice: %s", hipGetErrorString(err));
  KMOE_REQUIRE(dev >= 0 && dev < kMaxDevices, KMOE_ERR_UNSUPPORTED, "moe_forward_static: device %d (at most %d)", dev,
               kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) (void)hipGetLastError();
    KMOE_REQUIRE(cap == hipStreamCaptureStatusNone, KMOE_ERR_UNSUPPORTED,
                 "moe_forward_static: the built-in buffer's address on device %d is not known yet and this stream is "
                 "being captured: call kmoe_moe_forward or kmoe_moe_forward_static once outside the capture first",
                 dev);
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return fail(KMOE_ERR_LAUNCH, "moe_forward_static: hipGetSymbolAddress on device %d: %s", dev,
                  hipGetErrorString(err));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return KMOE_OK;
}

// Looks the address up on behalf of later captured calls; failures (a capture in progress, a runtime error) are
// left for kmoe_moe_forward_static to report.
void learn_static_workspace(hipStream_t stream) {
  static thread_local int known_dev = -1;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  if (dev == known_dev) return;
  void* p = nullptr;
  char saved[sizeof(g_error)];
  memcpy(saved, g_error, sizeof(saved));
  if (static_workspace(&p, stream) == KMOE_OK) known_dev = dev;
  else memcpy(g_error, saved, sizeof(saved));  // not this call's failure
}

}  // namespace

extern "C" int kmoe_moe_forward_static(const kmoe_moe_args* a, kmoe_stream_t stream) {
  kmoe_moe_layout L;
  if (int rc = kmoe_moe_workspace_layout(a, &L)) return rc;
  KMOE_REQUIRE(L.total_bytes <= static_cast<size_t>(KMOE_STATIC_WORKSPACE_BYTES), KMOE_ERR_WORKSPACE,
               "moe_forward_static: this shape needs %zu bytes of scratch, the built-in buffer holds %zu "
               "(use kmoe_moe_forward with a workspace of the caller's)",
               L.total_bytes, static_cast<size_t>(KMOE_STATIC_WORKSPACE_BYTES));
  void* ws = nullptr;
  if (int rc = static_workspace(&ws, as_stream(stream))) return rc;
  // every slot of the layout is written by the stage that owns it before anything reads it, so
  // the last call's contents need no clearing
  return moe_forward_impl(a, ws, KMOE_STATIC_WORKSPACE_BYTES, stream, false);  // no second stream: nothing is created here
}
