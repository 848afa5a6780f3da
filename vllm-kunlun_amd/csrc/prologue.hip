// What a layer call does before its first GEMM, but for the sort, in ONE launch: routing and, for the quantised formats, the
// quantisation of the activations (per token to int8, per group of 128 to fp8). The two are independent - both read
// the layer's inputs only - so the first workgroups route tokens while the rest quantise rows: on the decode path one
// launch of a few microseconds instead of two. The routing workgroups stay in front at every size: they are the
// long-lived ones (dealt in turn with the quantising ones the launch ends in a tail of routing waves: DeepSeek-V3
// prefill, 4096 tokens, 29 -> 35 us).
//
// The sort of the routed pairs was here, too, for larger batches: workgroups of 16 waves that count the pairs of the tokens
// they route, and a second launch that places them, both with a part of the quantisation. Layer, us, that / the sort in
// launches of its own: Qwen3 dims int8 2048 tokens 197.6 / 197.6, 3000 264.9 / 261.7, 4096 307.1 / 307.9, 8192 520.3 / 522.5, bf16 4096
// 431 / 426; 32 experts of [2048 x 4096], top 4, int8 4096 tokens 306.0 / 297.7, 8192 563 / 555.
#include "quant_body.h"
#include "routing_body.h"

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

enum class Quant { None, I8Wave, I8Block, Fp8, Fp8Two };  // I8Wave: rows of up to 2048 values, a wave each; Fp8Two: two groups a lane

template <int SLOTS, bool SIGMOID, Quant Q>
__global__ __launch_bounds__(256) void route_quant_kernel(const RouteArgs r, const QuantArgs q, int routing_blocks) {
  extern __shared__ float choice_lds[];  // sigmoid routing: [kWavesPerBlock][E]
  const int at = blockIdx.x;
  const int quant_at = at - routing_blocks;
  if (Q == Quant::None || at < routing_blocks) {
    const int wave = threadIdx.x >> 6, m = at * kWavesPerBlock + wave;
    if (m >= r.M) return;
    if constexpr (SIGMOID)
      sigmoid_group_topk_body<SLOTS>(r.logits, r.bias, m, r.E, r.K, r.n_group, r.topk_group, r.scale, r.topk_w, r.topk_ids,
                                     choice_lds + wave * r.E);
    else
      softmax_topk_body<SLOTS>(r.logits, m, r.E, r.K, r.renorm, r.topk_w, r.topk_ids);
  } else if (Q == Quant::I8Wave) {
    quant_i8_rows_body<64, 4>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, quant_at * 4, q.f16 != 0);
  } else if (Q == Quant::I8Block) {
    quant_i8_rows_body<256, 4>(q.x, q.ld_x, q.R, q.C, static_cast<int8_t*>(q.q), q.ld_q, q.aux, q.chunked, quant_at, q.f16 != 0);
  } else if (Q == Quant::Fp8 || Q == Quant::Fp8Two) {
    constexpr int NV = Q == Quant::Fp8Two ? 2 : 1;
    quant_fp8_group128_body<NV>(q.x, q.ld_x, q.R, q.C, static_cast<uint8_t*>(q.q), q.ld_q, q.aux, quant_at * (16u * NV), q.f16 != 0);
  }
}

template <int SLOTS, bool SIGMOID, Quant Q>
void launch(const RouteArgs& r, const QuantArgs& q, int quant_blocks, hipStream_t s) {
  const int routing_blocks = ceil_div(r.M, kWavesPerBlock);
  const size_t lds = SIGMOID ? sizeof(float) * kWavesPerBlock * r.E : 0;
  hipLaunchKernelGGL((route_quant_kernel<SLOTS, SIGMOID, Q>), dim3(routing_blocks + quant_blocks), dim3(256), lds, s, r,
                     q, routing_blocks);
}

long long fp8_groups(int rows, int values) { return static_cast<long long>(rows) * (values / 128); }

template <int SLOTS, bool SIGMOID>
void launch_q(const RouteArgs& r, const QuantArgs& q, Quant kind, hipStream_t s) {
  switch (kind) {
    case Quant::None: return launch<SLOTS, SIGMOID, Quant::None>(r, q, 0, s);
    case Quant::I8Wave: return launch<SLOTS, SIGMOID, Quant::I8Wave>(r, q, ceil_div(q.R, 4), s);
    case Quant::I8Block: return launch<SLOTS, SIGMOID, Quant::I8Block>(r, q, q.R, s);
    case Quant::Fp8: return launch<SLOTS, SIGMOID, Quant::Fp8>(r, q, static_cast<int>((fp8_groups(q.R, q.C) + 15) / 16), s);
    case Quant::Fp8Two: return launch<SLOTS, SIGMOID, Quant::Fp8Two>(r, q, static_cast<int>((fp8_groups(q.R, q.C) + 31) / 32), s);
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
                       bool chunked, bool f16, bool* quantised, hipStream_t s) {
  *quantised = false;
  if (int rc = check_route(&r, sigmoid)) return rc;
  Quant kind = Quant::None;
  if (format == KMOE_FMT_INT8 && H % 16 == 0 && H <= 256 * 8 * 4)  // wider rows: a launch of their own
    kind = H <= 64 * 8 * 4 ? Quant::I8Wave : Quant::I8Block;
  else if (format == KMOE_FMT_FP8_BLOCK && fp8_groups(r.M, H) < (1LL << 30))
    kind = fp8_groups(r.M, H) >= kFp8TwoGroups ? Quant::Fp8Two : Quant::Fp8;
  const QuantArgs q{x, H, r.M, H, xq, chunked ? 0 : H, x_aux, chunked ? 1 : 0, f16 ? 1 : 0};
  if (sigmoid) launch_e<true>(r, q, kind, s);
  else launch_e<false>(r, q, kind, s);
  *quantised = kind != Quant::None;
  return check_launch("kmoe_moe_forward (routing + quantisation)");
}

}  // namespace kmoe
