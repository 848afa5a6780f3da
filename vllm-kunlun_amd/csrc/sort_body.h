// What the launches that sort the routed pairs by expert share: keys, match ranks, the scan over the experts.
#pragma once
#include "kmoe_common.h"

namespace kmoe {

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

}  // namespace kmoe
