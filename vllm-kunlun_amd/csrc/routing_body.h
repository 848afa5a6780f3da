// Routing as device functions (one wave per token; expert e of the row lives in
// lane e % 64, slot e / 64), shared by the stand-alone routing kernels and the
// fused routing + activation-quantisation launch.
#pragma once
#include "kmoe_common.h"

namespace kmoe {

constexpr int kMaxSlots = 16;  // E <= 1024
constexpr int kWavesPerBlock = 4;

// Where scores are 16-bit values their patterns' 16 bits order them: bf16 in the upper half of the float's key; a half's own,
// made to an ordered key as ordered_bits does it (-0 as +0, NaNs quiet as the conversion to float leaves them).
__device__ inline uint32_t key_of_score(float score, int type, int id) {
  if (type == 0) return ordered_bits(score);
  uint32_t top;
  if (type == 1) {
    top = ordered_bits(score) >> 16;
  } else {
    const uint32_t h = __builtin_bit_cast(uint16_t, static_cast<_Float16>(score + 0.0f));
    top = (h & 0x8000u) ? ~h & 0xffffu : h | 0x8000u;
  }
  return (top << 16) | (0xffffu - static_cast<uint32_t>(id));
}
template <int CTRL>
__device__ inline float dpp_moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// The K best entries of the row held as key[s] (expert lane + 64 s; larger is better, 0: not a candidate) in K rounds
// of the largest key: rank[s] < K is the place of a chosen entry. A round finds its winner by comparing keys, on the vector
// unit alone - no ballot, whose way through the scalar unit was half of a round. Equal keys win a round together: returns
// how many entries have won then, with rank[s] the round, and 0 if every round had one winner.
template <int SLOTS>
__device__ inline int rank_topk(uint32_t (&key)[SLOTS], int K, int (&rank)[SLOTS]) {
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) rank[s] = K;
  uint32_t best;
  for (int k = 0; k < K; ++k) {
    best = 1;  // (never an entry that has won, or was none: all others may have gone in earlier rounds)
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) best = max(best, key[s]);
    best = group_max_u32<kWave>(best);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const bool won = key[s] == best;
      rank[s] = won ? k : rank[s];
      key[s] = won ? 0 : key[s];
    }
  }
  int chosen = 0;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) chosen += __builtin_popcountll(__ballot(rank[s] < K));
  const bool last = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(best)) > 1;  // the last round had a winner
  return chosen == K && last ? 0 : chosen;
}

// `from` and the lanes of the mask below this one.
__device__ inline int count_below(uint64_t lanes, int from) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(lanes >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(lanes), from));
}

// Picks the K best (score desc, expert id asc) entries of the row held as score[s] (expert lane + 64*s); lane k < K
// returns the k-th winner in my_id and its value[] in got. An entry's key is its score's order-preserving 32-bit pattern;
// where the scores are 16-bit values (`type` of LogitsView: 1 bf16, 2 half), which are often equal, the 16 bits that tell
// them apart and the id, so that no two keys are the same. The winners send id and value to their lanes.
// Equal keys are told apart behind the rounds, by round and id: float32 logits that a 16-bit gate left repeat as often as
// its own do. Launch, us, a ballot in every round / such tokens gone over a second time / so: softmax, 8 of 128 experts, 64
// tokens 3.36 / 3.63 / 3.08, 10 of 512 5.60 / 6.89 / 4.81, 32 of 1024 18.9 / 25.4 / 12.5, 8 of 128, 4096 tokens 4.33 / 5.33 / 4.44;
// sigmoid without a bias, 8 of 256, 64 tokens 3.70 / 4.46 / 3.51.
template <int SLOTS>
__device__ inline void select_topk(const float (&score)[SLOTS], const bool (&eligible)[SLOTS], const float (&value)[SLOTS], int type,
                                   int K, int lane, int& my_id, float& got) {
  uint32_t key[SLOTS];
  int rank[SLOTS];
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) key[s] = eligible[s] ? key_of_score(score[s], type, lane + kWave * s) : 0;
  if (const int won = rank_topk<SLOTS>(key, K, rank); won != 0) {
    if (won < kWave && won <= 2 * K) {  // side by side in the lanes, each counts those before it (a lane read per entry)
      uint32_t mine = 0;
      int at = 0, bits = 0;
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const bool chosen = rank[s] < K;
        const uint64_t here = __ballot(chosen);
        const int to = 4 * (chosen ? count_below(here, at) : kWave - 1);
        mine |= __builtin_amdgcn_ds_permute(to, chosen ? (rank[s] << 16) | (lane + kWave * s) : 0);
        bits |= __builtin_amdgcn_ds_permute(to, chosen ? __builtin_bit_cast(int, value[s]) : 0);
        at += __builtin_popcountll(here);
      }
      int place = 0;
      for (int i = 0; i < won; ++i) place += static_cast<uint32_t>(__builtin_amdgcn_readlane(mine, i)) < mine ? 1 : 0;
      const int to = 4 * (lane < won && place < K ? place : kWave - 1);
      my_id = __builtin_amdgcn_ds_permute(to, static_cast<int>(mine & 0xffffu));
      got = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(to, bits));
      return;
    }
    // many, or K = 64: round by round until there are K (a ballot per round and slot)
    int round[SLOTS], before = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      round[s] = rank[s];
      rank[s] = K;
    }
    for (int k = 0; k < K && before < K; ++k) {
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const uint64_t here = __ballot(round[s] == k);
        if (round[s] == k) rank[s] = min(count_below(here, before), K);
        before += __builtin_popcountll(here);
      }
    }
  }
  my_id = 0;
  int bits = 0;  // (entries that were not chosen send zeros to the last lane, which has no winner for K < 64)
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const bool chosen = rank[s] < K;
    const int to = 4 * (chosen ? rank[s] : kWave - 1);
    my_id |= __builtin_amdgcn_ds_permute(to, chosen ? lane + kWave * s : 0);
    bits |= __builtin_amdgcn_ds_permute(to, chosen ? __builtin_bit_cast(int, value[s]) : 0);
  }
  if (K == kWave) {
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const uint64_t last = __ballot(rank[s] == kWave - 1);
      if (last == 0) continue;
      const int from = __builtin_ctzll(last);
      const int v = __builtin_amdgcn_readlane(__builtin_bit_cast(int, value[s]), from);
      if (lane == kWave - 1) {
        my_id = from + kWave * s;
        bits = v;
      }
    }
  }
  got = __builtin_bit_cast(float, bits);
}

// p of lanes 0 ... K - 1 added in this order, in every lane.
__device__ inline float sum_in_order(float p, int K) {
  float sum = 0.0f;
  for (int k = 0; k < K; ++k) sum = sum + __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), k));
  return sum;
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

// One wave routes token m. weights: false leaves topk_w alone, for callers that ask only
// which experts a token goes to.
template <int SLOTS>
__device__ inline void softmax_topk_body(const LogitsView& logits, int m, int E, int K, int renorm,
                                         float* __restrict__ topk_w, int32_t* __restrict__ topk_ids, bool weights = true) {
  const int lane = lane_id();
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
  // exp and the row sum: per-lane running sum over slots, then the lane tree.
  float ex[SLOTS] = {};
  float total = 1.0f;
  if (weights) {
    mx = wave_max(mx);
    float part = 0.0f;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      ex[s] = ok[s] ? exp_fixed(v[s] - mx) : 0.0f;
      part = part + ex[s];
    }
    total = wave_sum_tree(part);
  }

  // lane k owns winner k and its exp
  int my_id;
  float got;
  select_topk<SLOTS>(v, ok, ex, logits.type, K, lane, my_id, got);
  if (lane < K) topk_ids[static_cast<size_t>(m) * K + lane] = my_id;
  if (!weights) return;
  float p = lane < K ? got / total : 0.0f;
  if (renorm) p = p / sum_in_order(p, K);  // k ascending
  if (lane < K) topk_w[static_cast<size_t>(m) * K + lane] = p;
}

// choice: E floats of the wave's own in LDS (groups that are no power of two, or longer than a wave).
template <int SLOTS>
__device__ inline void sigmoid_group_topk_body(const LogitsView& logits, const float* __restrict__ bias, int m,
                                               int E, int K, int n_group, int topk_group, float scale,
                                               float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
                                               float* choice, bool weights = true) {
  const int lane = lane_id();
  const size_t row = static_cast<size_t>(m) * E;

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
      // largest, all slots side by side
      float t1[SLOTS], t2[SLOTS];
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        t1[s] = fmaxf(c[s], -__builtin_inff());  // (a NaN counts as no score)
        t2[s] = -__builtin_inff();
      }
      // (steps of 1, 2, 4 ... lanes: once groups of N agree, the mirrored half row and row serve as lane l ^ N)
      auto merge = [&](auto other) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
          const float o1 = other(t1[s]), o2 = other(t2[s]);
          t2[s] = fmaxf(fminf(t1[s], o1), fmaxf(t2[s], o2));
          t1[s] = fmaxf(t1[s], o1);
        }
      };
      merge([](float v) { return dpp_moved<0xB1>(v); });                    // quad_perm [1,0,3,2]
      if (gsize >= 4) merge([](float v) { return dpp_moved<0x4E>(v); });    // quad_perm [2,3,0,1]
      if (gsize >= 8) merge([](float v) { return dpp_moved<0x141>(v); });   // row_half_mirror
      if (gsize >= 16) merge([](float v) { return dpp_moved<0x140>(v); });  // row_mirror
      if (gsize >= 32)
        merge([](float v) {
          const uint32_t u = __builtin_bit_cast(uint32_t, v);
          const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
          const uint32_t a = r[0], b = r[1];  // (chosen between as values, and nothing captured: elements and captured flags went over the stack)
          return __builtin_bit_cast(float, (lane_id() & 16) != 0 ? a : b);
        });
      if (gsize >= 64)
        merge([](float v) {
          const uint32_t u = __builtin_bit_cast(uint32_t, v);
          const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
          const uint32_t a = r[0], b = r[1];
          return __builtin_bit_cast(float, lane_id() >= 32 ? a : b);
        });
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        const float t = __shfl(t1[s] + t2[s], (lane * gsize) & (kWave - 1), kWave);
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
    // kept: the groups that fewer than topk_group others precede (score desc, group asc)
    const uint32_t gkey = lane < n_group ? ordered_bits(gscore) : 0;
    int ahead = 0;
    for (int g = 0; g < n_group; ++g) {
      const uint32_t other = __builtin_amdgcn_readlane(gkey, g);
      ahead += (other > gkey || (other == gkey && g < lane)) ? 1 : 0;
    }
    const uint64_t keep = __ballot(lane < n_group && ahead < topk_group);
    const int shift = (gsize & (gsize - 1)) == 0 ? __builtin_ctz(gsize) : -1;  // (a division takes some twenty instructions)
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      const int e = lane + kWave * s;
      const int group = shift >= 0 ? e >> shift : e / gsize;
      if (ok[s]) ok[s] = (keep >> group) & 1u;
    }
  }

  int my_id;
  float p;
  select_topk<SLOTS>(c, ok, sg, 0, K, lane, my_id, p);
  if (lane < K) topk_ids[static_cast<size_t>(m) * K + lane] = my_id;
  if (!weights) return;
  if (lane >= K) p = 0.0f;
  float denom = sum_in_order(p, K);
  denom = denom + 1e-20f;
  p = (p / denom) * scale;
  if (lane < K) topk_w[static_cast<size_t>(m) * K + lane] = p;
}

}  // namespace kmoe
