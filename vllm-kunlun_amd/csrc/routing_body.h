// Routing as device functions (one wave per token; expert e of the row lives in
// lane e % 64, slot e / 64), shared by the stand-alone routing kernels and the
// fused routing + activation-quantisation launch.
#pragma once
#include "kmoe_common.h"

namespace kmoe {

constexpr int kMaxSlots = 16;  // E <= 1024
constexpr int kWavesPerBlock = 4;

// Largest of a 32-bit value over the 64 lanes, in a scalar register: four DPP steps leave every 16-lane row with its
// own maximum, four lane reads and three scalar maxima do the rest.
__device__ inline uint32_t wave_max_u32(uint32_t v) {
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xB1, 0xf, 0xf, true)));   // quad_perm [1,0,3,2]
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4E, 0xf, 0xf, true)));   // quad_perm [2,3,0,1]
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xf, 0xf, true)));  // row_half_mirror
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x140, 0xf, 0xf, true)));  // row_mirror
  const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
  const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
  return max(max(a, b), max(c, d));
}

// Picks the K best (score desc, expert id asc) entries of the row held as
// score[s] (expert lane + 64*s); lane k < K returns the k-th winner in my_id.
// A score is its order-preserving 32-bit pattern (0: not a candidate); the round's winner is the lowest slot and
// lane that holds the maximum, found by ballots: a third of the instructions of a reduction on (score, id) pairs.
template <int SLOTS>
__device__ inline void select_topk(const float (&score)[SLOTS], const bool (&eligible)[SLOTS], int K,
                                   int lane, int& my_id) {
  uint32_t key[SLOTS];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) key[s] = eligible[s] ? ordered_bits(score[s]) : 0;
  my_id = -1;
  for (int k = 0; k < K; ++k) {
    uint32_t best = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) best = max(best, key[s]);
    best = wave_max_u32(best);
    int id = 0;
#pragma unroll
    for (int s = SLOTS - 1; s >= 0; --s) {
      const uint64_t holds = __ballot(key[s] == best);
      if (holds != 0) id = kWave * s + __builtin_ctzll(holds);
    }
    if (best == 0) id = -1;  // (fewer candidates than K: the host refuses such arguments)
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      if (id == lane + kWave * s) key[s] = 0;  // taken
    if (lane == k) my_id = id;
  }
}

// The row's logits, expert lane + 64 s in v[s]; experts past the last read the last one. Every load is requested
// before any is used: the routing waves of a decode batch are a few dependent memory round trips and little else.
template <int SLOTS>
__device__ inline void load_logits(const LogitsView& l, size_t row, int E, float (&v)[SLOTS]) {
  const int lane = lane_id();
  if (l.type != 0) {
    uint16_t h[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) h[s] = static_cast<const uint16_t*>(l.p)[row + min(lane + kWave * s, E - 1)];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) v[s] = act_to_f32(h[s], l.type == 2);
    return;
  }
  const float* at = static_cast<const float*>(l.p) + row;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) v[s] = at[min(lane + kWave * s, E - 1)];
  if (l.planes > 1) {  // at most 8 planes: request them all, then add in plane order
    float t[SLOTS][7];
#pragma unroll
    for (int p = 1; p < 8; ++p) {
      const float* plane = at + (p < l.planes ? p : 0) * l.plane_stride;
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) t[s][p - 1] = plane[min(lane + kWave * s, E - 1)];
    }
#pragma unroll
    for (int p = 1; p < 8; ++p)
#pragma unroll
      for (int s = 0; s < SLOTS; ++s)
        if (p < l.planes) v[s] = v[s] + t[s][p - 1];
  }
}

// One wave per token: workgroup `block` of kWavesPerBlock waves serves tokens
// block * kWavesPerBlock + wave.
template <int SLOTS>
__device__ inline void softmax_topk_body(const LogitsView& logits, int M, int E, int K, int renorm,
                                         float* __restrict__ topk_w, int32_t* __restrict__ topk_ids, int block) {
  const int lane = lane_id();
  const int m = block * kWavesPerBlock + (threadIdx.x >> 6);
  if (m >= M) return;
  const size_t row = static_cast<size_t>(m) * E;

  float v[SLOTS];
  bool ok[SLOTS];
  float mx = -__builtin_inff();
  load_logits<SLOTS>(logits, row, E, v);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    ok[s] = lane + kWave * s < E;
    v[s] = ok[s] ? v[s] : -__builtin_inff();
    mx = fmaxf(mx, v[s]);
  }
  mx = wave_max(mx);

  // exp and the row sum: per-lane running sum over slots, then the lane tree.
  float ex[SLOTS];
  float part = 0.0f;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    ex[s] = ok[s] ? exp_fixed(v[s] - mx) : 0.0f;
    part = part + ex[s];
  }
  const float total = wave_sum_tree(part);

  int my_id;
  select_topk<SLOTS>(v, ok, K, lane, my_id);

  // Lane k owns winner k: fetch its exp from the owning lane/slot.
  float p = 0.0f;
  {
    const int want = my_id >= 0 ? my_id : 0;
    float got = 0.0f;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const float t = __shfl(ex[s], want & (kWave - 1), kWave);
      if ((want >> 6) == s) got = t;
    }
    if (lane < K) p = got / total;
  }
  if (renorm) {
    float denom = 0.0f;
    for (int k = 0; k < K; ++k) denom = denom + __shfl(p, k, kWave);  // k ascending
    p = p / denom;
  }
  if (lane < K) {
    topk_w[static_cast<size_t>(m) * K + lane] = p;
    topk_ids[static_cast<size_t>(m) * K + lane] = my_id;
  }
}

// choice_lds: [kWavesPerBlock][E] floats of (dynamic) LDS.
template <int SLOTS>
__device__ inline void sigmoid_group_topk_body(const LogitsView& logits, const float* __restrict__ bias, int M,
                                               int E, int K, int n_group, int topk_group, float scale,
                                               float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
                                               float* choice_lds, int block) {
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  const int m = block * kWavesPerBlock + wave;
  if (m >= M) return;  // whole wave leaves together; no block-level sync below
  const size_t row = static_cast<size_t>(m) * E;
  float* choice = choice_lds + wave * E;

  float sg[SLOTS];  // un-biased sigmoid
  float c[SLOTS];   // score used for choosing
  bool ok[SLOTS];
  float bv[SLOTS];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) bv[s] = bias ? bias[min(lane + kWave * s, E - 1)] : 0.0f;
  load_logits<SLOTS>(logits, row, E, sg);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    ok[s] = lane + kWave * s < E;
    const float score = sigmoid_fixed(sg[s]);
    sg[s] = ok[s] ? score : 0.0f;
    c[s] = ok[s] ? (bias ? score + bv[s] : score) : -__builtin_inff();
  }

  if (n_group > 1) {
    const int gsize = E / n_group;
    // lane g < n_group: sum of the two largest scores of group g
    float gscore = -__builtin_inff();
    if ((gsize & (gsize - 1)) == 0 && gsize <= kWave) {
      // groups of 2 to 64 experts side by side in the lanes of a slot: a butterfly over the group keeps the two
      // largest (for 32 experts five exchanges where one lane walking the LDS copy of its group is a chain of 32
      // reads and compares: DeepSeek-V3 routing at 23 tokens 10.2 -> 6 us)
      float top[SLOTS];
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        float t1 = fmaxf(c[s], -__builtin_inff()), t2 = -__builtin_inff();  // (a NaN counts as no score)
        for (int off = gsize >> 1; off > 0; off >>= 1) {
          const float o1 = __shfl_xor(t1, off, kWave), o2 = __shfl_xor(t2, off, kWave);
          t2 = fmaxf(fminf(t1, o1), fmaxf(t2, o2));
          t1 = fmaxf(t1, o1);
        }
        top[s] = t1 + t2;
      }
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const float t = __shfl(top[s], (lane * gsize) & (kWave - 1), kWave);
        if (lane < n_group && (lane * gsize) / kWave == s) gscore = t;
      }
    } else {
#pragma unroll
      for (int s = 0; s < SLOTS; ++s)
        if (ok[s]) choice[lane + kWave * s] = c[s];
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own LDS writes have landed
      if (lane < n_group) {
        float t1 = -__builtin_inff(), t2 = -__builtin_inff();
        const float* gp = choice + lane * gsize;
        for (int i = 0; i < gsize; ++i) {
          const float x = gp[i];
          if (x > t1) {
            t2 = t1;
            t1 = x;
          } else if (x > t2) {
            t2 = x;
          }
        }
        gscore = t1 + t2;
      }
    }
    uint64_t keep = 0;
    uint32_t gkey = lane < n_group ? ordered_bits(gscore) : 0;
    for (int t = 0; t < topk_group; ++t) {
      const uint32_t best = wave_max_u32(gkey);
      const int bi = __builtin_ctzll(__ballot(gkey == best));  // the lowest group among equals
      if (bi == lane) gkey = 0;
      keep |= static_cast<uint64_t>(1) << (bi & 63);
    }
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const int e = lane + kWave * s;
      if (ok[s]) ok[s] = (keep >> (e / gsize)) & 1u;
    }
  }

  int my_id;
  select_topk<SLOTS>(c, ok, K, lane, my_id);

  float p = 0.0f;
  {
    const int want = my_id >= 0 ? my_id : 0;
    float got = 0.0f;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const float t = __shfl(sg[s], want & (kWave - 1), kWave);
      if ((want >> 6) == s) got = t;
    }
    if (lane < K) p = got;
  }
  float denom = 0.0f;
  for (int k = 0; k < K; ++k) denom = denom + __shfl(p, k, kWave);  // k ascending
  denom = denom + 1e-20f;
  p = (p / denom) * scale;
  if (lane < K) {
    topk_w[static_cast<size_t>(m) * K + lane] = p;
    topk_ids[static_cast<size_t>(m) * K + lane] = my_id;
  }
}


}  // namespace kmoe
