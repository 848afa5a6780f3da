// The layer of a few tokens in two launches.
//
// few_down_kernel: second quantisation, down projection and weighted combine.
//
// A batch of a few tokens is a chain of launches that each read a few MB: what it costs is launches and dependent memory
// round trips. In the down projection every routed pair is one row, so a workgroup can own 16 output channels of one TOKEN:
// a wave per routed expert (and one for the shared expert that rides along) streams that expert's 16 channels over all of K
// for the pair's row, the rows of the result meet in LDS, and the workgroup adds them up as the combine would - no launch
// that reads the down rows back, none for the quantisation in front: each wave quantises its own row while its weights are on
// their way. (Down rows, codes and their scales are still written, for whoever inspects the workspace; nothing here waits for
// them.) An expert that several tokens share is read once per token (from the caches), which is why this stops at a few of them.
#include <algorithm>

#include "buffer_ops.h"
#include "few_rows.h"
#include "formats.h"
#include "kmoe_common.h"
#include "quant_body.h"
#include "routing_body.h"
#include "w4_unpack.h"

namespace kmoe {
namespace {

// Whether a launch reads the weights that only one of its workgroups reads past the caches (see buffer_stream_load16): from 64 MB
// of pairs on. A layer called again at once with the same few experts finds fewer bytes in the 256 MB memory-side cache; with other
// layers' weights read in between they would gain from it too. Layer, us, ordinary / past the caches, called again at once; cold:
// DeepSeek-V3 dims int8, 1 token (235 MB in gate_up) 78.3 / 72.0, fp8 83.5 / 74.6, Kimi-K2 dims 4-bit (117 MB) 52.5 / 49.1; Qwen3 dims
// int8, 1 token (25 MB) 15.5 / 17.0; 19.5 / 18.5, 2 tokens (50 MB) 21.0 / 20.4; 24.0 / 22.5, bf16, 1 token (50 MB) 19.5 / 21.1; 24.4 / 23.3,
// 4-bit, 1 token (13 MB) 14.8 / 15.6; 17.9 / 16.9.
__device__ inline bool past_caches(size_t pairs, int channels, int row_bytes) {
  return pairs * channels * row_bytes > (64u << 20);
}

constexpr bool few_wide_i8(Fmt f, int vecs) { return f == Fmt::I8 && vecs > 2; }

// Steps of weights in flight (a multiple of the four chains; 4-bit, whose chains are a step's own: three, which hide the unpacking, are fewer
// registers than eight and less code to bring in, but eight - DEEP - where the launch has fewer waves than a row values, long rows and too few waves to
// keep the memory busy with three. Layer, time with three over time with eight, even load: Qwen3 dims 2 tokens 0.97, 6 0.96, Kimi-K2 dims 1 0.94, 160
// experts of [5120 x 1536] (hidden x intermediate), top 6, 1 0.97, 256 of [3072 x 512], top 8, 3 0.95, but 32 of [4096 x 2048], top 2, 1 to 4 tokens 1.05 / 1.02 /
// 1.01 / 1.01, 32 of [2048 x 1024], top 4, 1 and 2 1.03 / 1.02, 3 0.99, 64 of [4096 x 2048], top 8, 1 1.015, 2 0.97)
constexpr int few_down_steps(Fmt f, int vecs, bool deep) {
  return f == Fmt::W4 || f == Fmt::W4H ? (deep ? 8 : 3) : (f == Fmt::F8 ? 4 : (few_wide_i8(f, vecs) ? 12 : 8));
}
// kVecs: vectors of 8 values a lane holds of its row (rows of up to 512 kVecs values)
template <Fmt FMT, int kVecs, bool DEEP>
__global__ __launch_bounds__(kFewMaxWaves* kWave, few_wide_i8(FMT, kVecs) ? 4 : 5) void few_down_kernel(const FewDown p) {
  using acc_t = typename std::conditional<FMT == Fmt::I8, v4i, v4f>::type;
  constexpr bool W4 = FMT == Fmt::W4 || FMT == Fmt::W4H;
  constexpr bool QUANT = FMT == Fmt::I8 || FMT == Fmt::F8;
  constexpr int V = FMT == Fmt::F8 ? 2 : 1;   // 1 KB blocks of weights per step
  constexpr int AV = W4 ? 4 : V;              // 16-byte vectors of activations per lane and step ...
  constexpr int kAVStride = W4 ? 16 : 64, kALane = W4 ? 64 : 16, kAStep = W4 ? 256 : 64 * V;
  constexpr int D = few_down_steps(FMT, kVecs, DEEP);
  extern __shared__ __attribute__((aligned(16))) int8_t rows_lds[];  // [wave][few_row_pitch]
  __shared__ float y_lds[kFewMaxWaves][16];
  __shared__ float w_lds[kFewMaxWaves];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int m = blockIdx.y, col = blockIdx.x * 16;
  const bool f16 = FMT == Fmt::F16 || FMT == Fmt::W4H || ((FMT == Fmt::I8 || FMT == Fmt::F8) && p.f16 != 0);
  const bool tail = wave >= p.K;
  // (One token's waves could take the sorted rows 0 ... K - 1 and ask for them before they know whose they are. Layer, int8, so /
  // that way, us: Qwen3 dims 13.25 / 13.68, 64 experts of [3072 x 2560] 19.85 / 20.0, DeepSeek-V3 dims 67.5 / 67.1: the weights are asked for
  // later then, behind vector loads and a ballot where these three are scalar loads.)
  const int pair = m * p.K + wave;
  const int e = tail ? 0 : p.ids[pair];
  const int row = tail ? p.M * p.K + m : p.moe_index[pair];
  const float weight = tail ? 0.0f : p.topk_w[pair];

  // ---- weights: as many steps of the 16 channels as the ring holds ----
  const int ksteps = p.kbytes / (64 * V);
  const size_t frag_bytes = static_cast<size_t>(ksteps) * (V * 1024);
  const int8_t* w_base = (tail ? p.w_tail : p.w + static_cast<size_t>(e) * p.H * p.kbytes) + (col / 16) * frag_bytes;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(w_base), 0, static_cast<int>(frag_bytes), 0x00020000);
  // What the workgroups of several tokens read - an expert that several chose, the shared expert - is left to the caches. Layer,
  // us, past the caches all / as here, uniform routing cold; every token on the same eight experts, called again at once: Qwen3 dims int8 4
  // tokens 33.5 / 33.4; 19.3 / 19.2, 6 44.7 / 43.6; 23.0 / 21.6, 8 54.0 / 53.0; 27.2 / 24.4, 10 62.2 / 61.6; 29.1 / 26.3, bf16 4 54.6 / 53.6; 25.6 /
  // 22.5, 7 82.5 / 80.7; 34.5 / 27.0. (Uniform routing called again at once, 8 and 10 tokens: 52.4 / 52.8 and 60.4 / 61.5, with ordinary loads
  // alone 51.7 and 59.5, but cold 54.5 and 62.8: part of what is left to the caches is there from the call before.)
  bool past = past_caches(static_cast<size_t>(p.M) * p.K, p.H, p.kbytes);
  if (past && p.M > 1) {
    const int pairs = p.M * p.K;
    int readers = tail ? p.M : 0;
    if (!tail)
      for (int j = lane; j - lane < pairs; j += 2 * kWave) {  // (two loads at once: 128 pairs are a memory round trip)
        const int id[2] = {p.ids[min(j, pairs - 1)], p.ids[min(j + kWave, pairs - 1)]};
        readers += __builtin_popcountll(__ballot(j < pairs && id[0] == e)) + __builtin_popcountll(__ballot(j + kWave < pairs && id[1] == e));
      }
    past = readers == 1;
  }
  v4i wreg[D][V];
  uint16_t gsc[W4 ? D : 1];
  const uint16_t* sp = W4 ? p.w_scale + (static_cast<size_t>(e) * p.H + col) * p.groups + li * p.s_ch : nullptr;
  auto load_w = [&](int slot, int s) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const uint32_t at = static_cast<uint32_t>(s) * (V * 1024) + v * 1024;
      if (past) wreg[slot][v] = buffer_stream_load16(wr, lane * 16, at);
      else wreg[slot][v] = buffer_load16(wr, lane * 16, at);
    }
    if constexpr (W4) {
      const int g32 = 4 * s + lg;  // this lane's 32 values of the step
      gsc[slot] = sp[(p.gs_shift >= 0 ? g32 >> p.gs_shift : g32 / p.gs32) * p.s_g];
    }
  };
  float4 wmax = make_float4(0, 0, 0, 0);
  if constexpr (FMT == Fmt::I8) wmax = *reinterpret_cast<const float4*>((tail ? p.w_aux_tail : p.w_aux + static_cast<size_t>(e) * p.H) + col + lg * 4);
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < ksteps) load_w(d, d);
  float wsc = 0.0f;  // F8: lane l holds the block scale of step l
  if constexpr (FMT == Fmt::F8)
    wsc = (tail ? p.w_aux_tail : p.w_aux + static_cast<size_t>(e) * (p.H / 128) * ksteps)[static_cast<size_t>(col / 128) * ksteps + min(lane, ksteps - 1)];

  __builtin_amdgcn_sched_barrier(0);
  // ---- the row: quantised (the arithmetic of the quantisers' launches, hence their bits) or as it is, into LDS ----
  // (layer, us, loads under conditions / together: Qwen3 dims 3 tokens int8 24.75 / 24.5, fp8 25.8 / 25.5, DeepSeek-V3 dims fp8 1 token
  // 72.6 / 71.4; 16-bit and 4-bit rows, more registers and fewer waves, lose: bf16 4 tokens 48.4 / 53.9, Kimi-K2 dims 1 token 47.5 / 51.4)
  const uint4* src = reinterpret_cast<const uint4*>(p.act + static_cast<size_t>(row) * p.I);
  const int nvec = p.I / 8;
  Pack8 val[kVecs];
#pragma unroll
  for (int i = 0; i < kVecs; ++i) {
    if constexpr (QUANT) {  // lanes past the end read the last vector again: the loads go out together
      val[i].v = src[min(lane + i * kWave, nvec - 1)];
    } else {
      val[i].v = make_uint4(0, 0, 0, 0);
      if (lane + i * kWave < nvec) val[i].v = src[lane + i * kWave];
    }
  }
  int8_t* mine = rows_lds + wave * few_row_pitch(p.I, QUANT ? 1 : 2, FMT == Fmt::F8);
  [[maybe_unused]] float* scales = reinterpret_cast<float*>(mine + p.I);
  float amax = 1.0f;
  if constexpr (FMT == Fmt::I8) {
    uint32_t mag = 0;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) mag = max_magnitudes(mag, magnitudes8(val[i]));
    RowScale s = row_scale_i8(group_max_u32<kWave>(max_of_pair(mag)), f16);
    if (!s.numbers) {
      float top = 0.0f;
#pragma unroll
      for (int i = 0; i < kVecs; ++i) top = fmaxf(top, amax8(val[i], f16));
      s.amax = __builtin_bit_cast(float, group_max_u32<kWave>(__builtin_bit_cast(uint32_t, top)));
      s.inv = s.amax > 0.0f ? 127.0f / s.amax : 0.0f;
    }
    amax = s.amax;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int v = lane + i * kWave;
      if (v < nvec) {
        const uint2 codes = quant8_i8_of(val[i], s, f16);
        *reinterpret_cast<uint2*>(mine + v * 8) = codes;
        if (blockIdx.x == 0)  // what the quantiser's launch would have left
          *reinterpret_cast<uint2*>(p.codes + (static_cast<size_t>(v >> 3) * p.rows + row) * 64 + (v & 7) * 8) = codes;
      }
    }
    if (blockIdx.x == 0 && lane == 0) p.code_aux[row] = amax;
  } else if constexpr (FMT == Fmt::F8) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int v = lane + i * kWave;
      if (v < nvec) {  // (a group's 16 lanes together: nvec is a multiple of 16)
        float s;
        const uint2 codes = quant8_fp8(val[i], f16, s);
        *reinterpret_cast<uint2*>(mine + v * 8) = codes;
        if (blockIdx.x == 0) *reinterpret_cast<uint2*>(p.codes + static_cast<size_t>(row) * p.I + v * 8) = codes;
        if ((lane & 15) == 0) {
          scales[v >> 4] = s;
          if (blockIdx.x == 0) p.code_aux[static_cast<size_t>(row) * (p.I / 128) + (v >> 4)] = s;
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
      if (lane + i * kWave < nvec) *reinterpret_cast<uint4*>(mine + (lane + i * kWave) * 16) = val[i].v;
  }

  if constexpr (FMT == Fmt::I8) {  // (the scales' divisions while the weights come in)
    amax = amax / 127.0f;
    wmax = make_float4(wmax.x / 127.0f, wmax.y / 127.0f, wmax.z / 127.0f, wmax.w / 127.0f);
    asm("" : "+v"(amax), "+v"(wmax.x), "+v"(wmax.y), "+v"(wmax.z), "+v"(wmax.w));
  }

  // ---- product: all 16 rows of the MFMA are this row (its bytes are broadcast from LDS); four chains of sums ----
  acc_t acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = acc_t{0, 0, 0, 0};
  const int8_t* ap = mine + lg * kALane;
  for (int i0 = 0; i0 < ksteps; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int s = i0 + d;
      if (s < ksteps) {
        v4i av[AV];
#pragma unroll
        for (int v = 0; v < AV; ++v) av[v] = *reinterpret_cast<const v4i*>(ap + s * kAStep + v * kAVStride);
        acc_t& sum = acc[d & 3];
        if constexpr (FMT == Fmt::I8) {
          sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[d][0], av[0], sum, 0, 0, 0);
        } else if constexpr (FMT == Fmt::F8) {
          const float sw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wsc), s));
          const v4f blk = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              __builtin_shufflevector(wreg[d][0], wreg[d][V - 1], 0, 1, 2, 3, 4, 5, 6, 7),
              __builtin_shufflevector(av[0], av[V - 1], 0, 1, 2, 3, 4, 5, 6, 7), (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
          const float sc = scales[s] * sw;
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[q] = __builtin_fmaf(blk[q], sc, sum[q]);
        } else if constexpr (W4) {
          const W4Scale<FMT == Fmt::W4H> sc(gsc[W4 ? d : 0]);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const v4i wv = unpack8(static_cast<uint32_t>(wreg[d][0][t]), sc);
            if constexpr (FMT == Fmt::W4)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wv), __builtin_bit_cast(v8bf, av[AV > 1 ? t : 0]), acc[t], 0, 0, 0);
            else
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wv), __builtin_bit_cast(v8h, av[AV > 1 ? t : 0]), acc[t], 0, 0, 0);
          }
        } else if constexpr (FMT == Fmt::BF16) {
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wreg[d][0]), __builtin_bit_cast(v8bf, av[0]), sum, 0, 0, 0);
        } else {
          sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wreg[d][0]), __builtin_bit_cast(v8h, av[0]), sum, 0, 0, 0);
        }
        if (s + D < ksteps) load_w(d, s + D);
      }
    }
  }
  const acc_t total = (acc[0] + acc[1]) + (acc[2] + acc[3]);

  // ---- 16 channels of the pair's row, rounded as the down launch stores them; lanes 0, 16, 32, 48 hold four each ----
  if (li == 0) {
    uint16_t y[4];
    const float wm[4] = {wmax.x, wmax.y, wmax.z, wmax.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (FMT == Fmt::I8) y[q] = f32_to_act((static_cast<float>(total[q]) * amax) * wm[q], f16);
      else y[q] = f32_to_act(total[q], f16);
      y_lds[wave][lg * 4 + q] = act_to_f32(y[q], f16);
    }
    *reinterpret_cast<uint2*>(p.down + static_cast<size_t>(row) * p.H + col + lg * 4) =
        make_uint2(y[0] | (static_cast<uint32_t>(y[1]) << 16), y[2] | (static_cast<uint32_t>(y[3]) << 16));
    if (lane == 0) w_lds[wave] = weight;
  }
  __syncthreads();

  // ---- combine: f32 sum over the token's experts in routing order, one rounding, the caller's epilogue ----
  if (threadIdx.x < 16) {
    const int c = threadIdx.x;
    float sum = 0.0f;
    for (int k = 0; k < p.K; ++k) sum = __builtin_fmaf(w_lds[k], y_lds[k][c], sum);
    uint16_t o = f32_to_act(sum, f16);
    if (p.out_scale != 1.0f) o = f32_to_act(act_to_f32(o, f16) * p.out_scale, f16);
    if (p.w_tail) {
      float add = y_lds[p.K][c];
      if (p.shared_scale != 1.0f) add = act_to_f32(f32_to_act(add * p.shared_scale, f16), f16);
      o = f32_to_act(act_to_f32(o, f16) + add, f16);
    }
    p.out[static_cast<size_t>(m) * p.H + col + c] = o;
  }
}

// (the most rows there may be - 16 of 2048 16-bit values, 64.25 KB - fit a CU's 160 KB twice, with what the kernel holds besides)
static_assert(kFewMaxWaves * few_row_pitch(kFewMaxI, 2, false) + kFewMaxWaves * 17 * 4 <= 80 * 1024);
template <Fmt FMT, int kVecs, bool DEEP = false>
int launch_few_down(const FewDown& p, hipStream_t s) {
  const int waves = p.K + (p.w_tail ? 1 : 0);
  const size_t bytes = static_cast<size_t>(waves) * few_row_pitch(p.I, FMT == Fmt::I8 || FMT == Fmt::F8 ? 1 : 2, FMT == Fmt::F8);
  if (tracing_kernels())
    note_kernel("few_down_kernel<%s, %d steps in flight>, %d waves: quantisation, down projection and combine of a token's 16 channels", fmt_name(FMT),
                few_down_steps(FMT, kVecs, DEEP), waves);
  hipLaunchKernelGGL((few_down_kernel<FMT, kVecs, DEEP>), dim3(p.H / 16, p.M), dim3(waves * kWave), bytes, s, p);
  return check_launch("kmoe_moe_forward (down + combine)");
}

template <Fmt FMT>
int launch_few_down(const FewDown& p, hipStream_t s) {
  if constexpr (FMT == Fmt::W4 || FMT == Fmt::W4H) {
    if (static_cast<long long>(p.H / 16) * p.M * p.K <= p.I)
      return p.I <= 1024 ? launch_few_down<FMT, 2, true>(p, s) : launch_few_down<FMT, 4, true>(p, s);
  }
  return p.I <= 1024 ? launch_few_down<FMT, 2>(p, s) : launch_few_down<FMT, 4>(p, s);
}


// few_gate_up_kernel (up to kFewRouted tokens): routing, first quantisation, sort, gate_up projection and SiLU-mul.
//
// A workgroup serves 16 output channels of one routed PAIR's expert (columns of the grid: pairs, then the shared expert if
// one rides along, then one that leaves the routing and the sort for whoever reads them). It routes every token itself, a
// wave each, from the logits: a dozen cache lines and a microsecond against a launch of four before this one. (Which experts
// only: their weights are the last column's business.) The first
// pair that chose an expert serves all its rows; the other columns leave. The four waves split K; each quantises its own
// part of the rows while its weights are on their way (int8: one exchange of the maxima), and the codes wait in LDS.
// One token alone is routed by wave 0, and the others bring its row to LDS meanwhile - quantised, but for int8, whose scale
// is known only when all three have their part: each wave then rounds its part of K from there. Layer, us, the row asked for
// behind the weights / so: Qwen3 dims int8 14.75 / 13.7, fp8 15.1 / 14.7, bf16 19.0 / 18.8, 4-bit 13.7 / 13.5; DeepSeek-V3 dims int8 68.0 / 66.9,
// fp8 71.0 / 72.1; Kimi-K2 dims 4-bit 49.5 / 48.5.
// (The same for up to four tokens, every wave its part of all rows before the routing: 4 tokens 30.2 -> 33.3, a row then is
// looked at by every column and not by those that serve it.)
template <Fmt FMT, int SLOTS, bool SIGMOID>
__global__ __launch_bounds__(4 * kWave, FMT == Fmt::F8 ? 4 : 5) void few_gate_up_kernel(const FewGateUp p) {
  using acc_t = typename std::conditional<FMT == Fmt::I8, v4i, v4f>::type;
  constexpr bool W4 = FMT == Fmt::W4 || FMT == Fmt::W4H;
  constexpr bool QUANT = FMT == Fmt::I8 || FMT == Fmt::F8;
  constexpr int V = FMT == Fmt::F8 ? 2 : 1;
  constexpr int AV = W4 ? 4 : V;
  constexpr int kAVStride = W4 ? 16 : 64, kALane = W4 ? 64 : 16, kAStep = W4 ? 256 : 64 * V;
  constexpr int D = FMT == Fmt::F8 || W4 ? 2 : (FMT == Fmt::I8 ? 4 : 8);
  constexpr int kStepValues = W4 ? 128 : (QUANT ? 64 * V : 32);
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];  // sigmoid routing: [4][E] floats; then [M][few_row_pitch]
  __shared__ float tw_lds[kFewRouted * kFewMaxWaves];
  __shared__ int32_t id_lds[kFewRouted * kFewMaxWaves];
  __shared__ uint32_t max_lds[kFewRouted][4];
  __shared__ acc_t red[3][2][kWave];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const bool f16 = FMT == Fmt::F16 || FMT == Fmt::W4H || (QUANT && p.f16 != 0);
  const RouteArgs& r = p.route;
  const int P = r.M * r.K;
  const int column = blockIdx.y;
  const bool tail = p.w_tail != nullptr && column == P;
  const bool publish = column == P + (p.w_tail ? 1 : 0);
  if (publish && blockIdx.x != 0) return;
  const int pitch = few_row_pitch(p.H, QUANT ? 1 : 2, FMT == Fmt::F8);
  int8_t* const rows_lds = lds + (p.alone ? p.alone_at : 0);
  auto store_codes = [&](const Pack8& val, const RowScale& s, int8_t* dst, int v) __attribute__((always_inline)) {  // vector v of a row
    if constexpr (FMT == Fmt::I8) {
      *reinterpret_cast<uint2*>(dst + v * 8) = quant8_i8_of(val, s, f16);
    } else if constexpr (FMT == Fmt::F8) {
      float sc;
      *reinterpret_cast<uint2*>(dst + v * 8) = quant8_fp8(val, f16, sc);
      if ((lane & 15) == 0) reinterpret_cast<float*>(dst + p.H)[v >> 4] = sc;
    } else {
      *reinterpret_cast<uint4*>(dst + v * 16) = val.v;
    }
  };

  // ---- one token: waves 1 to 3 and its row ----
  if (p.alone && wave > 0 && !publish) {
    constexpr int kTakers = 3, kBatch = 5;  // (five vectors a lane: 7680 values in one round trip)
    uint32_t mag = 0;
    for (int v0 = (wave - 1) * kWave + lane; v0 - lane < p.H / 8; v0 += kBatch * kTakers * kWave) {
      Pack8 val[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        val[i].v = make_uint4(0, 0, 0, 0);
        if (v0 + i * kTakers * kWave < p.H / 8) val[i].v = reinterpret_cast<const uint4*>(p.x)[v0 + i * kTakers * kWave];
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int v = v0 + i * kTakers * kWave;
        if constexpr (FMT == Fmt::I8) {
          mag = max_magnitudes(mag, magnitudes8(val[i]));
          if (v < p.H / 8) *reinterpret_cast<uint4*>(rows_lds + pitch + v * 16) = val[i].v;
        } else {
          if (v < p.H / 8) store_codes(val[i], RowScale{}, rows_lds, v);
        }
      }
    }
    if constexpr (FMT == Fmt::I8) {
      mag = group_max_u32<kWave>(max_of_pair(mag));
      if (lane == 0) max_lds[0][wave] = mag;
    }
  }

  // ---- which expert, which rows ----
  int e = 0, rows = 0, begin = 0;
  int my_pair = 0;  // lane l: the pair of row l % 16 of this column
  if (!tail) {
    if (wave < r.M) {
      if constexpr (SIGMOID)
        sigmoid_group_topk_body<SLOTS>(r.logits, r.bias, wave, r.E, r.K, r.n_group, r.topk_group, r.scale, tw_lds, id_lds,
                                       reinterpret_cast<float*>(lds) + wave * r.E, publish);
      else
        softmax_topk_body<SLOTS>(r.logits, wave, r.E, r.K, r.renorm, tw_lds, id_lds, publish);
    }
    __syncthreads();
    const int id = lane < P ? id_lds[lane] : 0x7fffffff;  // (P <= 64)
    if (publish) {
      if (threadIdx.x < P) {
        r.topk_w[threadIdx.x] = tw_lds[threadIdx.x];
        r.topk_ids[threadIdx.x] = id;
        int below = 0, before = 0, equal = 0;  // pairs of lower experts; earlier pairs and all pairs of this one
        for (int j = 0; j < P; ++j) {
          below += id_lds[j] < id;
          before += id_lds[j] == id && j < static_cast<int>(threadIdx.x);
          equal += id_lds[j] == id;
        }
        p.sort.moe_index[threadIdx.x] = below + before;
        p.sort.sorted_src[below + before] = threadIdx.x;
        p.sort.slot_rows[threadIdx.x] = make_int2(below, before == 0 ? below + equal : below);  // (as scan_pairs leaves them)
      }
      for (int x = threadIdx.x; x < r.E; x += 4 * kWave) {
        int below = 0, equal = 0;
        for (int j = 0; j < P; ++j) {
          below += id_lds[j] < x;
          equal += id_lds[j] == x;
        }
        p.sort.lod[x] = below;
        p.sort.expert_m[x] = equal;
        if (x == r.E - 1) p.sort.lod[r.E] = below + equal;
      }
      return;
    }
    e = __builtin_amdgcn_readfirstlane(id_lds[column]);
    const uint64_t mine = __ballot(id == e);
    if (__builtin_ctzll(mine) != column) return;  // an earlier pair's column serves this expert
    rows = __builtin_popcountll(mine);            // (a token picks an expert once: at most kFewRouted)
    begin = __builtin_popcountll(__ballot(id < e));
    uint64_t left = mine;
#pragma unroll
    for (int i = 0; i < kFewRouted; ++i) {
      if (left != 0 && li == i) my_pair = __builtin_ctzll(left);
      left &= left - 1;
    }
  } else {
    rows = r.M;
    begin = P;
    if (p.alone) __syncthreads();
  }
  const int my_token = tail ? min(li, rows - 1) : my_pair / r.K;  // of row li (rows past the last: any token)

  // ---- weights of the gate and the up fragment: this wave's part of K, as many steps as the ring holds ----
  const int col = blockIdx.x * 16;
  const int ksteps = p.kbytes / (64 * V);
  const int kb0 = ksteps * wave / 4, klen = ksteps * (wave + 1) / 4 - kb0;
  const size_t frag_bytes = static_cast<size_t>(ksteps) * (V * 1024);
  const int8_t* w_base = tail ? p.w_tail : p.w + static_cast<size_t>(e) * (2 * p.I) * p.kbytes;
  __amdgpu_buffer_rsrc_t wr[2];
  const uint16_t* sp[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int c = f * p.I + col;
    wr[f] = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(w_base + (c / 16) * frag_bytes), 0, static_cast<int>(frag_bytes), 0x00020000);
    sp[f] = W4 ? p.w_scale + (static_cast<size_t>(e) * (2 * p.I) + c) * p.groups + li * p.s_ch : nullptr;
  }
  const bool past = past_caches(static_cast<size_t>(p.route.M) * p.route.K, 2 * p.I, p.kbytes);
  v4i wreg[D][2][V];
  uint16_t gsc[W4 ? D : 1][2];
  auto load_w = [&](int slot, int i) {
    const uint32_t s = kb0 + i;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const uint32_t at = s * (V * 1024) + v * 1024;
        if (past) wreg[slot][f][v] = buffer_stream_load16(wr[f], lane * 16, at);
        else wreg[slot][f][v] = buffer_load16(wr[f], lane * 16, at);
      }
      if constexpr (W4) {
        const int g32 = 4 * s + lg;
        gsc[slot][f] = sp[f][(p.gs_shift >= 0 ? g32 >> p.gs_shift : g32 / p.gs32) * p.s_g];
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < klen) load_w(d, d);
  float4 wmax[2];
  float wsc[2];  // F8: lane l holds the block scale of step kb0 + l
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int c = f * p.I + col;
    if constexpr (FMT == Fmt::I8)
      wmax[f] = *reinterpret_cast<const float4*>((tail ? p.w_aux_tail : p.w_aux + static_cast<size_t>(e) * (2 * p.I)) + c + lg * 4);
    if constexpr (FMT == Fmt::F8)
      wsc[f] = (tail ? p.w_aux_tail : p.w_aux + static_cast<size_t>(e) * (2 * p.I / 128) * ksteps)[static_cast<size_t>(c / 128) * ksteps + min(kb0 + lane, ksteps - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- the rows: this wave's part of K, quantised (the quantisers' arithmetic) or as it is, into LDS ----
  const int v0 = kb0 * (kStepValues / 8), nvec = klen * (kStepValues / 8);  // vectors of 8 values
  float amax = 1.0f;
  if constexpr (FMT == Fmt::I8) {
    for (int i = 0; i < rows && !p.alone; ++i) {
      const uint4* src = reinterpret_cast<const uint4*>(p.x + static_cast<size_t>(__builtin_amdgcn_readlane(my_token, i)) * p.H) + v0;
      uint32_t mag = 0;
      for (int v = lane; v < nvec; v += kWave) {
        Pack8 val;
        val.v = src[v];
        mag = max_magnitudes(mag, magnitudes8(val));
      }
      mag = group_max_u32<kWave>(max_of_pair(mag));
      if (lane == 0) max_lds[i][wave] = mag;
    }
    if (!p.alone) __syncthreads();
  }
  for (int i = 0; i < rows; ++i) {
    if (FMT != Fmt::I8 && p.alone) break;  // (done)
    const int token = __builtin_amdgcn_readlane(my_token, i);
    const uint4* src = reinterpret_cast<const uint4*>(p.x + static_cast<size_t>(token) * p.H);
    int8_t* dst = rows_lds + i * pitch;
    RowScale s = {};
    if constexpr (FMT == Fmt::I8) {
      s = row_scale_i8(max(max(p.alone ? 0u : max_lds[i][0], max_lds[i][1]), max(max_lds[i][2], max_lds[i][3])), f16);
      if (!s.numbers) {  // (the same for the whole workgroup) every wave goes over the whole row: rare
        float top = 0.0f;
        for (int v = lane; v < p.H / 8; v += kWave) {
          Pack8 val;
          val.v = src[v];
          top = fmaxf(top, amax8(val, f16));
        }
        s.amax = __builtin_bit_cast(float, group_max_u32<kWave>(__builtin_bit_cast(uint32_t, top)));
        s.inv = s.amax > 0.0f ? 127.0f / s.amax : 0.0f;
      }
      if (li == i) amax = s.amax;
      if (p.alone) {
        for (int v = lane; v < nvec; v += kWave) {
          Pack8 val;
          val.v = *reinterpret_cast<const uint4*>(rows_lds + pitch + (v0 + v) * 16);
          store_codes(val, s, dst, v0 + v);
        }
        break;
      }
    }
    for (int v = lane; v < nvec; v += kWave) {
      Pack8 val;
      val.v = src[v0 + v];
      store_codes(val, s, dst, v0 + v);
    }
  }

  // ---- product ----
  acc_t acc[2][2];
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[f][c] = acc_t{0, 0, 0, 0};
  const int8_t* arow = rows_lds + min(li, rows - 1) * pitch;
  const int8_t* ap = arow + lg * kALane + kb0 * kAStep;
  for (int i0 = 0; i0 < klen; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int i = i0 + d;
      if (i < klen) {
        v4i av[AV];
#pragma unroll
        for (int v = 0; v < AV; ++v) av[v] = *reinterpret_cast<const v4i*>(ap + i * kAStep + v * kAVStride);
        float sa = 1.0f;
        if constexpr (FMT == Fmt::F8) sa = reinterpret_cast<const float*>(arow + p.H)[kb0 + i];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          acc_t& sum = acc[f][d & 1];
          if constexpr (FMT == Fmt::I8) {
            sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[d][f][0], av[0], sum, 0, 0, 0);
          } else if constexpr (FMT == Fmt::F8) {
            const float sw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wsc[f]), i));
            const v4f blk = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                __builtin_shufflevector(wreg[d][f][0], wreg[d][f][V - 1], 0, 1, 2, 3, 4, 5, 6, 7),
                __builtin_shufflevector(av[0], av[V - 1], 0, 1, 2, 3, 4, 5, 6, 7), (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
            const float sc = sa * sw;
#pragma unroll
            for (int q = 0; q < 4; ++q) sum[q] = __builtin_fmaf(blk[q], sc, sum[q]);
          } else if constexpr (W4) {
            const W4Scale<FMT == Fmt::W4H> sc(gsc[W4 ? d : 0][f]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const v4i wv = unpack8(static_cast<uint32_t>(wreg[d][f][0][t]), sc);
              const v4i a = av[AV > 1 ? t : 0];
              if constexpr (FMT == Fmt::W4)
                acc[f][t & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wv), __builtin_bit_cast(v8bf, a), acc[f][t & 1], 0, 0, 0);
              else
                acc[f][t & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wv), __builtin_bit_cast(v8h, a), acc[f][t & 1], 0, 0, 0);
            }
          } else if constexpr (FMT == Fmt::BF16) {
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wreg[d][f][0]), __builtin_bit_cast(v8bf, av[0]), sum, 0, 0, 0);
          } else {
            sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wreg[d][f][0]), __builtin_bit_cast(v8h, av[0]), sum, 0, 0, 0);
          }
        }
        if (i + D < klen) load_w(d, i + D);
      }
    }
  }

  // ---- the four parts of K meet; SiLU-mul ----
  acc_t sum[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    sum[f] = acc[f][0] + acc[f][1];
    if (wave > 0) red[wave - 1][f][lane] = sum[f];
  }
  float sa = 1.0f;
  if constexpr (FMT == Fmt::I8) {  // (the divisions of the scales while the other waves come in)
    sa = amax / 127.0f;
    asm("" : "+v"(sa));
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      wmax[f] = make_float4(wmax[f].x / 127.0f, wmax[f].y / 127.0f, wmax[f].z / 127.0f, wmax[f].w / 127.0f);
      asm("" : "+v"(wmax[f].x), "+v"(wmax[f].y), "+v"(wmax[f].z), "+v"(wmax[f].w));
    }
  }
  __syncthreads();
  if (wave == 0 && li < rows) {
    uint16_t g[4], u[4];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
      for (int part = 0; part < 3; ++part) sum[f] += red[part][f][lane];
      const float wm[4] = {wmax[f].x, wmax[f].y, wmax[f].z, wmax[f].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint16_t& o = f == 0 ? g[q] : u[q];
        if constexpr (FMT == Fmt::I8) o = f32_to_act((static_cast<float>(sum[f][q]) * sa) * wm[q], f16);
        else o = f32_to_act(sum[f][q], f16);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] = f32_to_act(silu_hw(act_to_f32(g[q], f16)) * act_to_f32(u[q], f16), f16);
    *reinterpret_cast<uint2*>(p.act + static_cast<size_t>(begin + li) * p.I + col + lg * 4) =
        make_uint2(g[0] | (static_cast<uint32_t>(g[1]) << 16), g[2] | (static_cast<uint32_t>(g[3]) << 16));
  }
}

template <Fmt FMT, int SLOTS, bool SIGMOID>
int launch_few_gate_up(FewGateUp p, hipStream_t s) {
  const int pitch = few_row_pitch(p.H, FMT == Fmt::I8 || FMT == Fmt::F8 ? 1 : 2, FMT == Fmt::F8);
  // LDS: routing's copy of the scores, then the rows in its place; one token: beside that of the wave that routes it, with
  // the row as it is behind its codes (int8), if that leaves the five workgroups of few_gate_up_takes their room
  const size_t scores = SIGMOID ? sizeof(float) * p.route.E : 0;
  size_t bytes = std::max(static_cast<size_t>(p.route.M) * pitch, 4 * scores);
  const size_t alone = align_up(scores, 16) + pitch + (FMT == Fmt::I8 ? 2 * static_cast<size_t>(p.H) : 0);
  p.alone = p.route.M == 1 && alone <= kFewRowBytes;
  p.alone_at = static_cast<int32_t>(align_up(scores, 16));
  if (p.alone) bytes = alone;
  if (tracing_kernels())
    note_kernel("few_gate_up_kernel<%s>: routing, quantisation, sort and gate_up of a pair's 16 channels", fmt_name(FMT));
  hipLaunchKernelGGL((few_gate_up_kernel<FMT, SLOTS, SIGMOID>), dim3(p.I / 16, p.route.M * p.route.K + (p.w_tail ? 1 : 0) + 1), dim3(4 * kWave), bytes, s, p);
  return check_launch("kmoe_moe_forward (routing + gate_up)");
}

template <Fmt FMT>
int launch_few_gate_up(const FewGateUp& p, bool sigmoid, hipStream_t s) {
  const int slots = ceil_div(p.route.E, kWave);
  if (slots <= 2) return sigmoid ? launch_few_gate_up<FMT, 2, true>(p, s) : launch_few_gate_up<FMT, 2, false>(p, s);
  if (slots <= 4) return sigmoid ? launch_few_gate_up<FMT, 4, true>(p, s) : launch_few_gate_up<FMT, 4, false>(p, s);
  return sigmoid ? launch_few_gate_up<FMT, 8, true>(p, s) : launch_few_gate_up<FMT, 8, false>(p, s);
}

}  // namespace

int few_down(const FewDown& p, int format, hipStream_t s) {
  switch (format) {
    case KMOE_FMT_INT8: return launch_few_down<Fmt::I8>(p, s);
    case KMOE_FMT_FP8_BLOCK: return launch_few_down<Fmt::F8>(p, s);
    case KMOE_FMT_BF16: return p.f16 ? launch_few_down<Fmt::F16>(p, s) : launch_few_down<Fmt::BF16>(p, s);
    default: return p.f16 ? launch_few_down<Fmt::W4H>(p, s) : launch_few_down<Fmt::W4>(p, s);
  }
}

int few_gate_up(const FewGateUp& p, int format, bool sigmoid, hipStream_t s) {
  switch (format) {
    case KMOE_FMT_INT8: return launch_few_gate_up<Fmt::I8>(p, sigmoid, s);
    case KMOE_FMT_FP8_BLOCK: return launch_few_gate_up<Fmt::F8>(p, sigmoid, s);
    case KMOE_FMT_BF16: return p.f16 ? launch_few_gate_up<Fmt::F16>(p, sigmoid, s) : launch_few_gate_up<Fmt::BF16>(p, sigmoid, s);
    default: return p.f16 ? launch_few_gate_up<Fmt::W4H>(p, sigmoid, s) : launch_few_gate_up<Fmt::W4>(p, sigmoid, s);
  }
}

}  // namespace kmoe
