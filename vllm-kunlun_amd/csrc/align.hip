// moe_align: stable counting sort of routed pairs by expert id, built from LDS
// histograms, a per-expert scan and wavefront ballot ranks.
//
// Decomposition: the P pairs are cut into chunks of kThreads*steps consecutive pairs,
// one workgroup each; inside a chunk wave w owns the next kWave*steps pairs.
// The sorted row of pair j with expert e is
//   lod[e] + (#pairs of e in earlier chunks) + (#pairs of e in earlier waves /
//   steps of this chunk) + (#lower lanes of this step with expert e),
// which is exactly the stable order (ties by ascending j).
#include "kmoe_common.h"

namespace kmoe {
namespace {

constexpr int kThreads = 1024;            // workgroup size of the multi-workgroup kernels
constexpr int kWaves = kThreads / kWave;  // 16
constexpr int kMaxE = 1024;
// Launches by the number of pairs. One workgroup of 256 threads and cheap barriers up to 256 pairs and experts (3.3 us a
// call in a row of calls; 4.1 by the next). One launch of P / 1024 workgroups that each count every pair, us behind a launch
// that writes the ids, 256 experts: 4.0 at 512 pairs, 4.9 at 4096, 5.1 at 8192, 6.1 at 16384, 7.0 at 24000, 7.9 at 32768 (one
// workgroup for all took 4.5 at 512 and 9.1 at 4096). Two launches beyond, where reading all the ids in every workgroup costs
// more than the second launch: 9.4 at 32768 pairs and some 2 more with other kernels around, 9.5 at 49152 and 65536 (one: 9.8,
// 11.6), 22 at 2^20. Counting in every workgroup is what few experts, or few that most pairs go to, make slow (atomics on the
// same counters): beyond kNoWorkspaceMaxP pairs one launch from 64 experts on. One / two there, us with the ids' launch, 28000
// pairs: 8 experts 11.5 / 10.0, 16 10.2 / 10.4, 32 9.5 / 10.5, 64 9.6 / 11.0, 256 10.0 / 11.9, 1024 11.2 / 14.9; half of the pairs on a sixteenth
// of the experts: 8 18.9 / 10.2, 32 13.6 / 10.4, 64 11.4 / 10.7, 128 10.4 / 11.3, 256 9.8 / 11.6.
constexpr int kSingleMaxP = 256, kSingleMaxE = 256;
// Pairs beyond which callers have to bring a workspace, by their number alone (one launch does not look at it).
constexpr int kNoWorkspaceMaxP = 24576;
inline bool takes_one_launch(int P, int E) { return P <= kNoWorkspaceMaxP || (P <= 32768 && E >= 64); }
constexpr int kMaxChunks = 128;           // workgroups of the two-launch path at most

// two-launch path: pairs per thread
inline int chunk_steps(int P) { return max(2, ceil_div(P, kMaxChunks * kThreads)); }

__device__ inline int key_bits(int E) { return 32 - __builtin_clz(max(E - 1, 1)); }

// Rank of this lane among the lower lanes holding the same key, and the number
// of lanes holding it. Lanes with key < 0 are idle. One ballot per key bit: the
// lanes whose key agrees with mine on every bit are the lanes with my key.
__device__ inline void wave_match_rank(int key, int bits, int& rank, int& count) {
  const bool live = key >= 0;
  uint64_t same = __ballot(live);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (key >> b) & 1;
    const uint64_t set = __ballot(live && bit);
    same &= bit ? set : ~set;
  }
  rank = live ? __builtin_popcountll(same & lanemask_lt()) : 0;
  count = live ? __builtin_popcountll(same) : 0;
}

// The expert ids of the routed pairs as the routing kernel wrote them, seen by a launch that owns the experts
// [first, first + E) of them (an expert-parallel share; first = 0: all of them): ids outside come out outside [0, E).
struct IdView {
  const int32_t* ids;
  int first;
  __device__ int operator[](int j) const { return ids[j] - first; }
};

// The key of an id: its expert, or -1 (ids outside [0,E), pairs past the end: no sorted row).
__device__ inline int key_of(int id, int first, bool live, int E) {
  const int e = id - first;
  return live && static_cast<unsigned>(e) < static_cast<unsigned>(E) ? e : -1;
}
__device__ inline int load_key(const IdView ids, int j, int end, int E) {
  return j < end ? key_of(ids.ids[j], ids.first, true, E) : -1;
}

// Counting phase for one chunk: wave w owns pairs [begin + w*64*steps, +64*steps).
// Leaves in wcnt[w][e] the number of expert-e pairs of this chunk in waves < w and
// returns to thread e < E the chunk's total for expert e (0 to the other threads).
// `wcnt` is LDS scratch [waves][E].
__device__ inline int count_chunk(const IdView ids, int begin, int end, int E, int steps,
                                  int* wcnt) {
  const int waves = blockDim.x >> 6;
  const int wave = threadIdx.x >> 6;
  const int lane = lane_id();
  const int bits = key_bits(E);
  const int wbegin = begin + wave * kWave * steps;
  for (int i = threadIdx.x; i < waves * E; i += blockDim.x) wcnt[i] = 0;
  __syncthreads();
  int* mine = wcnt + wave * E;
  for (int s = 0; s < steps; ++s) {
    const int key = load_key(ids, wbegin + s * kWave + lane, end, E);
    int rank, count;
    wave_match_rank(key, bits, rank, count);
    if (key >= 0 && rank == 0) mine[key] += count;  // one lane per distinct expert; a wave's LDS ops stay in order
  }
  __syncthreads();
  int total = 0;
  for (int e = threadIdx.x; e < E; e += blockDim.x) {  // at most one trip: blockDim.x >= E
    for (int w = 0; w < waves; ++w) {
      const int c = wcnt[w * E + e];
      wcnt[w * E + e] = total;
      total += c;
    }
  }
  return total;
}

// Scatter phase: pair j of expert e lands at base[e] + wcnt[wave][e] + (rank among the
// wave's earlier pairs of e). Call after count_chunk and a barrier that publishes base.
__device__ inline void scatter_chunk(const IdView ids, int begin, int end, int E, int steps,
                                     const int* base, int* wcnt, int32_t* __restrict__ moe_index,
                                     int32_t* __restrict__ sorted_src) {
  const int wave = threadIdx.x >> 6;
  const int lane = lane_id();
  const int bits = key_bits(E);
  const int wbegin = begin + wave * kWave * steps;
  int* mine = wcnt + wave * E;
  for (int s = 0; s < steps; ++s) {
    const int j = wbegin + s * kWave + lane;
    const int key = load_key(ids, j, end, E);
    int rank, count;
    wave_match_rank(key, bits, rank, count);
    if (j < end && key < 0) moe_index[j] = -1;
    if (key >= 0) {
      const int pos = base[key] + mine[key] + rank;
      moe_index[j] = pos;
      if (sorted_src) sorted_src[pos] = j;
    }
    __builtin_amdgcn_wave_barrier();
    if (key >= 0 && rank == 0) mine[key] += count;
    __builtin_amdgcn_wave_barrier();
  }
}

// Exclusive scan of cnt[0..E) by one workgroup (blockDim.x >= E): a shuffle scan
// inside each wave, then the wave totals through LDS. Writes lod[0..E] and
// expert_m (where they are given), and leaves lod[e] also in out_base[e]. `wtot` is LDS scratch of 16 ints.
__device__ inline void scan_experts(int my_count /* thread e < E */, int E, int* wtot, int* out_base,
                                    int32_t* __restrict__ lod, int32_t* __restrict__ expert_m) {
  const int t = threadIdx.x;
  const int lane = lane_id();
  int incl = t < E ? my_count : 0;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  if (lane == kWave - 1) wtot[t >> 6] = incl;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < (t >> 6); ++w) before += wtot[w];
  if (t < E) {
    const int excl = before + incl - my_count;
    out_base[t] = excl;
    if (lod) lod[t] = excl;
    if (expert_m) expert_m[t] = my_count;
    if (lod && t == E - 1) lod[E] = before + incl;
  }
  __syncthreads();
}

// One workgroup of 256 threads, one pair each (P <= kSingleMaxP, E <= kSingleMaxE).
__global__ __launch_bounds__(kSingleMaxP) void align_single_kernel(
    const IdView ids, int P, int E, int32_t* __restrict__ moe_index,
    int32_t* __restrict__ sorted_src, int32_t* __restrict__ expert_m, int32_t* __restrict__ lod) {
  extern __shared__ int lds[];
  int* wtot = lds;          // [16]
  int* base = wtot + 16;    // [E]
  int* wcnt = base + E;     // [waves][E]
  const int mine = count_chunk(ids, 0, P, E, 1, wcnt);
  scan_experts(mine, E, wtot, base, lod, expert_m);
  scatter_chunk(ids, 0, P, E, 1, base, wcnt, moe_index, sorted_src);
}

// One launch for several workgroups (takes_one_launch): workgroup b owns the kThreads pairs of chunk b, one per
// thread, and counts ALL the pairs itself - those of earlier chunks apart from the rest - so that it knows where its
// chunk begins in every expert without waiting for another workgroup. Bound by latencies: a launch, the round trip of
// the ids, the barriers and the scan. kBatch loads in flight per thread: past the end the last id is read again, as loads
// under conditions of their own went out one after another (256 experts: 8192 pairs 7.2 -> 5.1 us, 24000 12.1 -> 7.0). Two
// where that is all of them, eight beyond (2048 pairs: 4.1, with eight 4.7; 16384 6.1, with sixteen 6.2).
template <int kBatch>
__global__ __launch_bounds__(kThreads) void align_one_launch_kernel(
    const IdView ids, int P, int E, int32_t* __restrict__ moe_index, int32_t* __restrict__ sorted_src,
    int32_t* __restrict__ expert_m, int32_t* __restrict__ lod) {
  extern __shared__ int lds[];
  int* wtot = lds;           // [16]
  int* base = wtot + 16;     // [E]
  int* before = base + E;    // [E]: pairs of earlier chunks
  int* rest = before + E;    // [E]: the others
  int* wcnt = rest + E;      // [kWaves][E]
  const int t = threadIdx.x, wave = t >> 6;
  const int begin = blockIdx.x * kThreads;
  auto id_at = [&](int j) { return ids.ids[max(min(j, P - 1), 0)]; };
  const int my_id = id_at(begin + t);
  int v[kBatch];
  auto load = [&](int j0) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = id_at(j0 + i * kThreads + t);
  };
  load(0);
  for (int i = t; i < (2 + kWaves) * E; i += kThreads) before[i] = 0;
  __syncthreads();
  const int key = key_of(my_id, ids.first, begin + t < P, E);
  int rank, count;
  wave_match_rank(key, key_bits(E), rank, count);
  if (key >= 0 && rank == 0) wcnt[wave * E + key] = count;
  for (int j0 = 0; j0 < P; j0 += kBatch * kThreads) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int e = key_of(v[i], ids.first, j0 + i * kThreads + t < P, E);
      if (e >= 0) atomicAdd((j0 + i * kThreads < begin ? before : rest) + e, 1);  // (chunks are whole: uniform)
    }
    load(j0 + kBatch * kThreads);
  }
  __syncthreads();
  int earlier = 0, total = 0;
  if (t < E) {
    earlier = before[t];
    total = earlier + rest[t];
    int mine = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int c = wcnt[w * E + t];
      wcnt[w * E + t] = mine;
      mine += c;
    }
  }
  scan_experts(total, E, wtot, base, blockIdx.x == 0 ? lod : nullptr, blockIdx.x == 0 ? expert_m : nullptr);
  if (begin + t >= P) return;
  if (key < 0) {
    moe_index[begin + t] = -1;
    return;
  }
  const int pos = base[key] + before[key] + wcnt[wave * E + key] + rank;
  moe_index[begin + t] = pos;
  if (sorted_src) sorted_src[pos] = begin + t;
}

// Two launches for more pairs than that, chunks of `steps` x kThreads pairs. Kernel 1: chunk histograms ->
// hist[chunk][E].
__global__ __launch_bounds__(kThreads) void align_hist_kernel(const IdView ids, int P, int E, int steps,
                                                             int32_t* __restrict__ hist) {
  extern __shared__ int lds[];
  for (int e = threadIdx.x; e < E; e += kThreads) lds[e] = 0;
  __syncthreads();
  const int begin = blockIdx.x * steps * kThreads;
  const int end = min(P, begin + steps * kThreads);
  for (int j = begin + threadIdx.x; j < end; j += kThreads) {
    const int e = load_key(ids, j, end, E);
    if (e >= 0) atomicAdd(&lds[e], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kThreads) hist[static_cast<size_t>(blockIdx.x) * E + e] = lds[e];
}

// Kernel 2: stable scatter of each chunk. Every workgroup sums the (at most kMaxChunks) histograms itself, the earlier
// chunks' apart: kThreads / E threads per expert, eight loads in flight each.
__global__ __launch_bounds__(kThreads) void align_scatter_kernel(const IdView ids, int P, int E, int steps, int n_chunks,
                                                                const int32_t* __restrict__ hist,
                                                                int32_t* __restrict__ moe_index,
                                                                int32_t* __restrict__ sorted_src,
                                                                int32_t* __restrict__ expert_m, int32_t* __restrict__ lod) {
  extern __shared__ int lds[];
  int* wtot = lds;         // [16]
  int* base = wtot + 16;   // [E]
  int* before = base + E;  // [E]: pairs of earlier chunks
  int* rest = before + E;  // [E]: the others
  int* wcnt = rest + E;    // [kWaves][E]
  const int t = threadIdx.x, me = blockIdx.x;
  for (int i = t; i < 2 * E; i += kThreads) before[i] = 0;
  const int begin = me * steps * kThreads;
  const int end = min(P, begin + steps * kThreads);
  count_chunk(ids, begin, end, E, steps, wcnt);  // (its barriers publish the zeros)
  const int parts = kThreads / E, part = t / E, e = t - part * E;
  if (part < parts) {
    constexpr int kBatch = 8;
    int lo = 0, hi = 0;
    for (int c0 = part; c0 < n_chunks; c0 += kBatch * parts) {
      int v[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int c = c0 + i * parts;
        v[i] = hist[static_cast<size_t>(min(c, n_chunks - 1)) * E + e];
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int c = c0 + i * parts;
        (c < me ? lo : hi) += c < n_chunks ? v[i] : 0;
      }
    }
    if (lo) atomicAdd(&before[e], lo);
    if (hi) atomicAdd(&rest[e], hi);
  }
  __syncthreads();
  scan_experts(t < E ? before[t] + rest[t] : 0, E, wtot, base, me == 0 ? lod : nullptr, me == 0 ? expert_m : nullptr);
  if (t < E) base[t] += before[t];
  __syncthreads();
  scatter_chunk(ids, begin, end, E, steps, base, wcnt, moe_index, sorted_src);
}

__global__ void block_statistic_kernel(const int32_t* __restrict__ ids, int P, int E, int per_block,
                                       int32_t* __restrict__ out) {
  extern __shared__ int lds[];
  for (int e = threadIdx.x; e < E; e += blockDim.x) lds[e] = 0;
  __syncthreads();
  const int begin = blockIdx.x * per_block;
  const int end = min(P, begin + per_block);
  for (int j = begin + threadIdx.x; j < end; j += blockDim.x) {
    const int e = ids[j];
    if (e >= 0 && e < E) atomicAdd(&lds[e], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) out[static_cast<size_t>(blockIdx.x) * E + e] = lds[e];
}

__global__ void gather_rows_kernel(const uint16_t* __restrict__ src, int64_t ld_src,
                                   const int32_t* __restrict__ sorted_src, int K, int H,
                                   uint16_t* __restrict__ dst, int64_t ld_dst) {
  const int r = blockIdx.x;
  const int tok = sorted_src[r] / K;
  const uint4* s = reinterpret_cast<const uint4*>(src + static_cast<size_t>(tok) * ld_src);
  uint4* d = reinterpret_cast<uint4*>(dst + static_cast<size_t>(r) * ld_dst);
  for (int i = threadIdx.x; i < H / 8; i += blockDim.x) d[i] = s[i];
}

}  // namespace
}  // namespace kmoe

using namespace kmoe;

extern "C" size_t kmoe_align_workspace_bytes(int P, int E) {
  if (P <= kNoWorkspaceMaxP || E <= 0) return 256;  // unused, but never report zero
  return align_up(static_cast<size_t>(ceil_div(P, chunk_steps(P) * kThreads)) * E * sizeof(int32_t), 256);
}

extern "C" int kmoe_align(const int32_t* topk_ids, int P, int E, int32_t* moe_index, int32_t* sorted_src,
                          int32_t* expert_m, int32_t* lod, void* workspace, size_t workspace_bytes,
                          kmoe_stream_t stream) {
  return kmoe_align_local(topk_ids, P, E, 0, moe_index, sorted_src, expert_m, lod, workspace, workspace_bytes, stream);
}

extern "C" int kmoe_align_local(const int32_t* ids_global, int P, int E, int first_expert, int32_t* moe_index,
                                int32_t* sorted_src, int32_t* expert_m, int32_t* lod, void* workspace,
                                size_t workspace_bytes, kmoe_stream_t stream) {
  const IdView topk_ids{ids_global, first_expert};
  KMOE_REQUIRE(first_expert >= 0, KMOE_ERR_SHAPE, "align: first_expert=%d", first_expert);
  KMOE_REQUIRE(lod && (P == 0 || (ids_global && moe_index)), KMOE_ERR_NULL, "align: NULL pointer");
  KMOE_REQUIRE(E >= 1 && E <= kMaxE, KMOE_ERR_SHAPE, "align: E=%d outside [1,%d]", E, kMaxE);
  KMOE_REQUIRE(P >= 0 && P <= (1 << 24), KMOE_ERR_SHAPE, "align: P=%d outside [0,2^24]", P);
  hipStream_t s = as_stream(stream);
  if (P <= kSingleMaxP && E <= kSingleMaxE) {
    const size_t lds = sizeof(int) * (16 + E + static_cast<size_t>(kSingleMaxP / kWave) * E);
    hipLaunchKernelGGL(align_single_kernel, dim3(1), dim3(kSingleMaxP), lds, s, topk_ids, P, E, moe_index, sorted_src,
                       expert_m, lod);
    return check_launch("kmoe_align");
  }
  const int steps = chunk_steps(P), n_chunks = ceil_div(P, steps * kThreads);
  const size_t need = static_cast<size_t>(n_chunks) * E * sizeof(int32_t);
  if (P > kNoWorkspaceMaxP) {
    KMOE_REQUIRE(workspace, KMOE_ERR_WORKSPACE, "align: workspace is NULL (need %zu bytes)", need);
    KMOE_REQUIRE(workspace_bytes >= need, KMOE_ERR_WORKSPACE, "align: workspace %zu < %zu bytes", workspace_bytes,
                 need);
  }
  if (takes_one_launch(P, E)) {
    const IdView some{P > 0 ? ids_global : lod, first_expert};  // (of no pairs: memory to read, whatever it holds)
    hipLaunchKernelGGL((P <= 2 * kThreads ? align_one_launch_kernel<2> : align_one_launch_kernel<8>), dim3(max(1, ceil_div(P, kThreads))),
                       dim3(kThreads), sizeof(int) * (16 + (3 + static_cast<size_t>(kWaves)) * E), s, some, P, E, moe_index, sorted_src,
                       expert_m, lod);
    return check_launch("kmoe_align");
  }
  int32_t* hist = static_cast<int32_t*>(workspace);
  hipLaunchKernelGGL(align_hist_kernel, dim3(n_chunks), dim3(kThreads), sizeof(int) * E, s, topk_ids, P, E, steps, hist);
  hipLaunchKernelGGL(align_scatter_kernel, dim3(n_chunks), dim3(kThreads),
                     sizeof(int) * (16 + (3 + static_cast<size_t>(kWaves)) * E), s, topk_ids, P, E, steps, n_chunks, hist,
                     moe_index, sorted_src, expert_m, lod);
  return check_launch("kmoe_align");
}

extern "C" int kmoe_block_statistic(const int32_t* topk_ids, int P, int E, int n_blocks,
                                    int32_t* block_statistic, kmoe_stream_t stream) {
  KMOE_REQUIRE(topk_ids && block_statistic, KMOE_ERR_NULL, "block_statistic: NULL pointer");
  KMOE_REQUIRE(E >= 1 && E <= 8192, KMOE_ERR_SHAPE, "block_statistic: E=%d outside [1,8192]", E);
  KMOE_REQUIRE(P >= 0 && n_blocks >= 1, KMOE_ERR_SHAPE, "block_statistic: P=%d n_blocks=%d", P, n_blocks);
  const int per_block = max(1, ceil_div(P, n_blocks));
  hipLaunchKernelGGL(block_statistic_kernel, dim3(n_blocks), dim3(256), sizeof(int) * E, as_stream(stream),
                     topk_ids, P, E, per_block, block_statistic);
  return check_launch("kmoe_block_statistic");
}

extern "C" int kmoe_gather_rows(const uint16_t* src, int64_t ld_src, const int32_t* sorted_src, int P, int K,
                                int H, uint16_t* dst, int64_t ld_dst, kmoe_stream_t stream) {
  KMOE_REQUIRE(src && sorted_src && dst, KMOE_ERR_NULL, "gather_rows: NULL pointer");
  KMOE_REQUIRE(P >= 0 && K >= 1 && H >= 8 && H % 8 == 0, KMOE_ERR_SHAPE, "gather_rows: P=%d K=%d H=%d", P, K, H);
  KMOE_REQUIRE(ld_src % 8 == 0 && ld_dst % 8 == 0 && ld_src >= H && ld_dst >= H, KMOE_ERR_SHAPE,
               "gather_rows: row strides %lld/%lld must be multiples of 8 and >= H", (long long)ld_src,
               (long long)ld_dst);
  if (P == 0) return KMOE_OK;
  hipLaunchKernelGGL(gather_rows_kernel, dim3(P), dim3(256), 0, as_stream(stream), src, ld_src, sorted_src, K, H,
                     dst, ld_dst);
  return check_launch("kmoe_gather_rows");
}
