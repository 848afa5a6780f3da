// What a layer call does before its first GEMM: routing, the sort of the routed pairs by expert and, for the quantised
// formats, the quantisation of the activations (per token to int8, per group of 128 to fp8).
//
// Decode batches, whose gate_up launch sorts: ONE launch, the first workgroups route tokens while the rest quantise rows - the
// two are independent, both read the layer's inputs only. The routing workgroups stay in front at every size: they are the
// long-lived ones (dealt in turn with the quantising ones the launch ends in a tail of routing waves: DeepSeek-V3
// prefill, 4096 tokens, 29 -> 35 us).
//
// Larger batches over up to 128 experts: TWO launches of workgroups of 1024. In the first a routing workgroup serves a chunk of
// 16, 32, 48 or 64 tokens, a wave each or several in turn, and leaves how many of its pairs went to each expert; in the second a
// workgroup per chunk adds those counts up and writes its pairs' places. The rows are quantised beside them, in either launch.
// Against the sort in one launch that counts all the pairs in every workgroup, or in two of its own beyond 32768 pairs, layer, us: Qwen3
// dims int8 1024 tokens 145.9 -> 146.8, 1500 175.0 both, 2048 194.4 -> 192.3, 4096 290.9 -> 289.3, 8192 521.3 -> 517.5, bf16 2048 286.5 ->
// 287.2, so from 12288 pairs on. Routing is bound by issue: 256 chunks, on all CUs, cost the second launch what they
// save the first (8192 tokens 523 to 527). More experts take longer to route: DeepSeek-V3 dims 1000 tokens 1944 / 1941, 4096 2569 / 2580,
// Kimi-K2 dims 2048 2423 / 2424: those keep the launches above and a sort behind them.
#include "quant_body.h"
#include "routing_body.h"
#include "sort_body.h"

namespace kmoe {
namespace {

struct QuantArgs {
  const uint16_t* x;
  int64_t ld_x;
  int R, C;
  void* q;
  int64_t ld_q;
  float* aux;  // int8: row maxes; fp8: group scales
  int chunked;
  int f16;
};

enum class Quant { None, I8Wave, I8Block, Fp8, Fp8Two };  // I8Wave: rows of up to 2048 values, a wave each; Fp8Two: two groups a lane (the launch that does not sort)

template <int SLOTS, bool SIGMOID>
__device__ inline int route_token(const RouteArgs& r, int m, float* choice) {
  if constexpr (SIGMOID)
    return sigmoid_group_topk_body<SLOTS>(r.logits, r.bias, m, r.E, r.K, r.n_group, r.topk_group, r.scale, r.topk_w, r.topk_ids, choice);
  else
    return softmax_topk_body<SLOTS>(r.logits, m, r.E, r.K, r.renorm, r.topk_w, r.topk_ids);
}

template <int SLOTS, bool SIGMOID, Quant Q>
__global__ __launch_bounds__(256) void route_quant_kernel(const RouteArgs r, const QuantArgs q, int routing_blocks) {
  extern __shared__ float choice_lds[];  // sigmoid routing: [kWavesPerBlock][E]
  const int at = blockIdx.x;
  const int quant_at = at - routing_blocks;
  if (Q == Quant::None || at < routing_blocks) {
    const int wave = threadIdx.x >> 6, m = at * kWavesPerBlock + wave;
    if (m < r.M) route_token<SLOTS, SIGMOID>(r, m, choice_lds + wave * r.E);
  } else if (Q == Quant::I8Wave) {
    quant_i8_rows_body<64, 4>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, quant_at * 4, q.f16 != 0);
  } else if (Q == Quant::I8Block) {
    quant_i8_rows_body<256, 4>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, quant_at, q.f16 != 0);
  } else if (Q == Quant::Fp8 || Q == Quant::Fp8Two) {
    constexpr int NV = Q == Quant::Fp8Two ? 2 : 1;
    quant_fp8_group128_body<NV>(q.x, q.ld_x, q.R, q.C, static_cast<uint8_t*>(q.q), q.ld_q, q.aux, quant_at * (16u * NV), q.f16 != 0);
  }
}

// ---- two launches ----
constexpr int kSortThreads = 1024, kSortWaves = kSortThreads / kWave;
constexpr int kSortSlots = 2;      // experts routed over / 64
constexpr int kSortChunks = 128;   // chunks at most, whose counts every workgroup of the second launch adds up
// Rows a workgroup of either launch quantises: a wave each up to 2048 values, four waves each beyond (fp8: groups of 128, 64 a workgroup).
constexpr int sort_rows(Quant q) { return q == Quant::I8Wave ? kSortWaves : kSortWaves / 4; }

struct SortArgs {
  SortOut out;
  const int32_t* ids;
  int P, K, tokens, chunks;  // tokens of a chunk, a multiple of kSortWaves; chunks
};

// Part `at` of q's rows (fp8: of their groups).
template <Quant Q>
__device__ inline void quantise_part(const QuantArgs& q, int at) {
  if constexpr (Q == Quant::I8Wave)
    quant_i8_rows_body<64, 4, kSortThreads>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, at * sort_rows(Q), q.f16 != 0);
  else if constexpr (Q == Quant::I8Block)
    quant_i8_rows_body<256, 4, kSortThreads>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, at * sort_rows(Q), q.f16 != 0);
  else if constexpr (Q == Quant::Fp8)
    quant_fp8_group128_body<1, kSortThreads>(q.x, q.ld_x, q.R, q.C, static_cast<uint8_t*>(q.q), q.ld_q, q.aux, at * (kSortThreads / 16u), q.f16 != 0);
}

// Workgroup c < s.chunks: chunk c's tokens routed, and its counts per expert (of those this launch owns) in s.out.counts.
template <int SLOTS, bool SIGMOID, Quant Q>
__global__ __launch_bounds__(kSortThreads) void route_count_quant_kernel(const RouteArgs r, const SortArgs s, const QuantArgs q) {
  extern __shared__ int count_lds[];  // [experts owned]; sigmoid routing, where it needs them: [kSortWaves][E] scores
  const int at = blockIdx.x;
  if (at >= s.chunks) return quantise_part<Q>(q, at - s.chunks);
  const int wave = threadIdx.x >> 6, lane = lane_id(), E = s.out.E;
  for (int e = threadIdx.x; e < E; e += kSortThreads) count_lds[e] = 0;
  __syncthreads();
  for (int i = wave; i < s.tokens; i += kSortWaves) {
    const int m = at * s.tokens + i;
    if (m >= r.M) break;
    const int id = route_token<SLOTS, SIGMOID>(r, m, reinterpret_cast<float*>(count_lds + E) + wave * r.E) - s.out.first;
    if (lane < r.K && static_cast<unsigned>(id) < static_cast<unsigned>(E)) atomicAdd(&count_lds[id], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kSortThreads) s.out.counts[static_cast<size_t>(at) * E + e] = count_lds[e];
}

// Workgroup c < s.chunks: the places of chunk c's pairs (one a thread) in the stable order by expert: behind lower experts' pairs,
// earlier chunks' of the same expert, and earlier ones of the chunk.
template <Quant Q>
__global__ __launch_bounds__(kSortThreads) void sort_quant_kernel(const SortArgs s, const QuantArgs q, int quant_from) {
  extern __shared__ int sort_lds[];
  if (static_cast<int>(blockIdx.x) >= s.chunks) return quantise_part<Q>(q, quant_from + blockIdx.x - s.chunks);
  const int E = s.out.E, me = blockIdx.x, t = threadIdx.x, wave = t >> 6;
  const int chunk = s.tokens * s.K, waves = (chunk + kWave - 1) / kWave;
  int* const wtot = sort_lds;          // [16]
  int* const base = wtot + 16;         // [E]
  int* const before = base + E;        // [E]: pairs of earlier chunks
  int* const rest = before + E;        // [E]: the others
  int* const wcnt = rest + E;          // [waves][E]
  const int begin = me * chunk, end = min(s.P, begin + chunk);
  const int key = load_key(IdView{s.ids, s.out.first}, begin + t, end, E);
  // counts: kSortThreads / E threads per expert, kBatch loads in flight each
  constexpr int kBatch = 16;
  const int parts = kSortThreads / E, part = t / E, e = t - part * E;
  const bool adds = part < parts;
  int v[kBatch];
  auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int c = c0 + i * parts;
      v[i] = s.out.counts[static_cast<size_t>(min(c, s.chunks - 1)) * E + e];
    }
  };
  load(part);
  for (int i = t; i < (2 + waves) * E; i += kSortThreads) before[i] = 0;
  __syncthreads();
  int rank = 0, count = 0;
  if (wave < waves) {
    wave_match_rank(key, key_bits(E), rank, count);
    if (key >= 0 && rank == 0) wcnt[wave * E + key] = count;
  }
  int lo = 0, hi = 0;
  for (int c0 = part; adds && c0 < s.chunks; c0 += kBatch * parts) {
    if (c0 != part) load(c0);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int c = c0 + i * parts;
      (c < me ? lo : hi) += c < s.chunks ? v[i] : 0;
    }
  }
  if (lo) atomicAdd(&before[e], lo);
  if (hi) atomicAdd(&rest[e], hi);
  __syncthreads();
  int total = 0;
  if (t < E) {
    total = before[t] + rest[t];
    int mine = 0;
    for (int w = 0; w < waves; ++w) {
      const int c = wcnt[w * E + t];
      wcnt[w * E + t] = mine;
      mine += c;
    }
  }
  scan_experts(total, E, wtot, base, me == 0 ? s.out.lod : nullptr, me == 0 ? s.out.expert_m : nullptr);
  if (begin + t >= end) return;
  if (key < 0) {
    s.out.moe_index[begin + t] = -1;
    return;
  }
  const int pos = base[key] + before[key] + wcnt[wave * E + key] + rank;
  s.out.moe_index[begin + t] = pos;
  s.out.sorted_src[pos] = begin + t;
}

template <int SLOTS, bool SIGMOID, Quant Q>
void launch(const RouteArgs& r, const QuantArgs& q, int quant_blocks, hipStream_t s) {
  const int routing_blocks = ceil_div(r.M, kWavesPerBlock);
  const size_t lds = SIGMOID ? sizeof(float) * kWavesPerBlock * r.E : 0;
  hipLaunchKernelGGL((route_quant_kernel<SLOTS, SIGMOID, Q>), dim3(routing_blocks + quant_blocks), dim3(256), lds, s, r,
                     q, routing_blocks);
}

template <int SLOTS, bool SIGMOID>
void launch_q(const RouteArgs& r, const QuantArgs& q, Quant kind, hipStream_t s) {
  switch (kind) {
    case Quant::None: return launch<SLOTS, SIGMOID, Quant::None>(r, q, 0, s);
    case Quant::I8Wave: return launch<SLOTS, SIGMOID, Quant::I8Wave>(r, q, ceil_div(q.R, 4), s);
    case Quant::I8Block: return launch<SLOTS, SIGMOID, Quant::I8Block>(r, q, q.R, s);
    case Quant::Fp8:
    case Quant::Fp8Two: {
      const long long groups = static_cast<long long>(q.R) * (q.C / 128);
      if (groups >= kFp8TwoGroups) return launch<SLOTS, SIGMOID, Quant::Fp8Two>(r, q, static_cast<int>((groups + 31) / 32), s);
      return launch<SLOTS, SIGMOID, Quant::Fp8>(r, q, static_cast<int>((groups + 15) / 16), s);
    }
  }
}

// Floats of LDS a routing wave needs for its scores.
int score_floats(const RouteArgs& r, bool sigmoid) {
  const int g = sigmoid && r.n_group > 1 ? r.E / r.n_group : 1;
  return (g & (g - 1)) != 0 || g > kWave ? r.E : 0;
}

// Whether a batch is sorted by the launches that route it: sizes that gain (above), a pair per thread, room for the counts.
bool sorts_with_routing(const RouteArgs& r, const SortArgs& s) {
  return s.P > 12288 && r.E <= kSortSlots * kWave && s.tokens <= 4 * kSortWaves && s.tokens * s.K <= kSortThreads &&
         static_cast<size_t>(s.chunks) * s.out.E * sizeof(int32_t) <= s.out.counts_bytes;
}

template <bool SIGMOID, Quant Q>
int launch_sorting(const RouteArgs& r, const SortArgs& s, const QuantArgs& q, int parts, hipStream_t st) {
  const int E = s.out.E;
  const size_t route_lds = sizeof(int) * (E + static_cast<size_t>(kSortWaves) * score_floats(r, SIGMOID));
  const size_t sort_lds = sizeof(int) * (16 + (3 + static_cast<size_t>(ceil_div(s.tokens * s.K, kWave))) * E);
  const int first = parts * 3 / 4;  // parts of the quantisation in the first launch (none to all of them: 517 to 525 us at 8192 tokens)
  hipLaunchKernelGGL((route_count_quant_kernel<kSortSlots, SIGMOID, Q>), dim3(s.chunks + first), dim3(kSortThreads), route_lds, st, r, s, q);
  if (int rc = check_launch("kmoe_moe_forward (routing + counts + quantisation)")) return rc;
  hipLaunchKernelGGL((sort_quant_kernel<Q>), dim3(s.chunks + parts - first), dim3(kSortThreads), sort_lds, st, s, q, first);
  return check_launch("kmoe_moe_forward (sort + quantisation)");
}

template <bool SIGMOID>
int launch_sorting(const RouteArgs& r, const SortArgs& s, const QuantArgs& q, Quant kind, hipStream_t st) {
  switch (kind) {
    case Quant::None: return launch_sorting<SIGMOID, Quant::None>(r, s, q, 0, st);
    case Quant::I8Wave: return launch_sorting<SIGMOID, Quant::I8Wave>(r, s, q, ceil_div(q.R, sort_rows(kind)), st);
    case Quant::I8Block: return launch_sorting<SIGMOID, Quant::I8Block>(r, s, q, ceil_div(q.R, sort_rows(kind)), st);
    default:
      return launch_sorting<SIGMOID, Quant::Fp8>(
          r, s, q, static_cast<int>((static_cast<long long>(q.R) * (q.C / 128) + kSortThreads / 16 - 1) / (kSortThreads / 16)), st);
  }
}

template <bool SIGMOID>
void launch_e(const RouteArgs& r, const QuantArgs& q, Quant kind, hipStream_t s) {
  const int slots = ceil_div(r.E, kWave);
  if (slots <= 2) launch_q<2, SIGMOID>(r, q, kind, s);
  else if (slots <= 4) launch_q<4, SIGMOID>(r, q, kind, s);
  else if (slots <= 8) launch_q<8, SIGMOID>(r, q, kind, s);
  else launch_q<16, SIGMOID>(r, q, kind, s);
}

}  // namespace

int check_route(RouteArgs* route, bool sigmoid) {
  RouteArgs& r = *route;
  KMOE_REQUIRE(r.E >= 1 && r.E <= kMaxSlots * kWave && r.K >= 1 && r.K <= r.E && r.K <= kWave, KMOE_ERR_SHAPE,
               "routing: E=%d K=%d", r.E, r.K);
  if (sigmoid) {
    if (r.n_group <= 1) {
      r.n_group = 1;
      r.topk_group = 1;
    } else {
      KMOE_REQUIRE(r.n_group <= kWave, KMOE_ERR_SHAPE, "routing: n_group=%d > 64", r.n_group);
      KMOE_REQUIRE(r.E % r.n_group == 0, KMOE_ERR_SHAPE, "routing: E=%d not divisible by n_group=%d", r.E, r.n_group);
      KMOE_REQUIRE(r.E / r.n_group >= 2, KMOE_ERR_SHAPE, "routing: groups of %d experts; need >= 2", r.E / r.n_group);
      KMOE_REQUIRE(r.topk_group >= 1 && r.topk_group <= r.n_group, KMOE_ERR_SHAPE,
                   "routing: topk_group=%d outside [1,n_group=%d]", r.topk_group, r.n_group);
      KMOE_REQUIRE(r.K <= r.topk_group * (r.E / r.n_group), KMOE_ERR_SHAPE,
                   "routing: K=%d exceeds the %d experts of the kept groups", r.K, r.topk_group * (r.E / r.n_group));
    }
  }
  return KMOE_OK;
}

int route_and_quantise(RouteArgs r, bool sigmoid, int format, const uint16_t* x, int H, void* xq, float* x_aux,
                       bool chunked, bool f16, const SortOut* sort, bool* quantised, bool* sorted, hipStream_t s) {
  *quantised = *sorted = false;
  if (int rc = check_route(&r, sigmoid)) return rc;
  Quant kind = Quant::None;
  if (format == KMOE_FMT_INT8 && H % 16 == 0 && H <= 256 * 8 * 4)  // wider rows: a launch of their own
    kind = H <= 64 * 8 * 4 ? Quant::I8Wave : Quant::I8Block;
  else if (format == KMOE_FMT_FP8_BLOCK && static_cast<long long>(r.M) * (H / 128) < (1LL << 30))
    kind = Quant::Fp8;
  const QuantArgs q{x, H, r.M, H, xq, chunked ? 0 : H, x_aux, chunked ? 1 : 0, f16 ? 1 : 0};
  *quantised = kind != Quant::None;
  if (sort) {
    SortArgs a{*sort, r.topk_ids, r.M * r.K, r.K, kSortWaves * ceil_div(r.M, kSortWaves * kSortChunks), 0};
    a.chunks = ceil_div(r.M, a.tokens);
    if (sorts_with_routing(r, a)) {
      *sorted = true;
      return sigmoid ? launch_sorting<true>(r, a, q, kind, s) : launch_sorting<false>(r, a, q, kind, s);
    }
  }
  if (sigmoid) launch_e<true>(r, q, kind, s);
  else launch_e<false>(r, q, kind, s);
  return check_launch("kmoe_moe_forward (routing + quantisation)");
}

}  // namespace kmoe
