// Dense W8A8 GEMM of a few rows (a Linear's decode and small-prefill batches): y[r, c] = sum_k a[r, k] w[c, k], weights
// tiled, activations chunk-major, int32 sums, dequantised at the end.
//
// A matrix of a few thousand channels has neither experts nor row tiles enough to fill 256 CUs, so what bounds it is
// latency: the bytes a CU has to fetch, over the bytes it keeps on their way. Both are set by the workgroup's shape here:
//   eight waves share ONE tile of 16 MF rows x 16 NF channels and split K eight ways, straight from memory to registers -
//   no LDS and no barrier in the main loop - with D steps of (NF + MF) KB in flight per wave, up to 144 KB per CU
//   (deeper rings gained nothing: from there on it is the bytes a CU takes in, about 40 a clock, that count);
//   a squarer tile means fewer bytes: [100 x 7168] x [4096 x 7168] takes 256 workgroups (one per CU) of 64 x 32 that
//   fetch 0.6 MB each, where slices of 32 rows with K split four ways fetched 0.9 MB per CU, 64 KB at a time.
// Rows are split evenly over the row tiles and rows past a tile's end are out of the descriptor's range: no bytes.
// The weights are read with ordinary loads: a Linear that is called again at once finds them in the 256 MB memory-side cache. With
// other layers' weights read in between, loads past the caches (see buffer_stream_load16) would be ahead while one row tile holds
// all rows. [4096 x 7168], SiLU-mul, [7168 x 2048], us, ordinary / past the caches, called again at once; cold: 1 row 14.8 / 14.7; 18.2 /
// 17.0, 16 21.2 / 22.7; 25.5 / 23.9, 100 29.0 / 31.9; 35.6 / 34.3, 200 35.6 / 40.6; 41.6 / 43.0. Up to four rows, too, smaller matrices
// lose: [1536 x 2048], SiLU-mul, [2048 x 768] 1 row 9.6 / 10.4; 11.2 / 10.9.
// The eight partial sums meet in LDS once; wave w then finishes fragments w, w + 8, ... of the tile. int32 sums are exact,
// so neither the split nor the order shows in a bit.
#include "buffer_ops.h"
#include "kmoe_common.h"
#include "quant_body.h"

namespace kmoe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

struct DenseParams {
  const int8_t* a;  // chunk-major [k/64][a_rows][64]
  int32_t a_rows, src0;
  const float* a_max;
  const uint16_t* x;  // QUANT: [rows, k] bf16 / half values, row stride ld_x, instead of a and a_max
  int64_t ld_x;
  const int8_t* w;  // tiled [n/16][k/64] blocks of 1 KB
  const float* w_max;
  int32_t n, k, rows, row0;  // output rows [row0, row0 + rows) read activation rows [src0, src0 + rows)
  int32_t tile_rows;
  uint16_t* y;
  int64_t ldy;
  int32_t* acc_out;
  int32_t f16;
  int32_t rotate;  // waves start their K range at a step of their own (rotates(k))
};

constexpr int kDenseWaves = 8;
// Whether the GEMM's launch quantises a few rows itself: every workgroup does, so a second row wants all of them on the chip at once, two
// per CU, and one row a launch of a few rounds (kQuantCost). With the quantiser's launch / in the GEMM's, us, called again at once; cold:
// [4096 x 7168] 1 row 11.9 / 8.5; 14.1 / 11.6, 4 rows 11.1 / 9.9; 14.4 / 16.3, [14336 x 4096] (448 workgroups) 1 13.8 / 11.5; 17.6 / 14.7, 4 13.8 /
// 14.3; 17.7 / 17.7, [8192 x 8192] 4 16.2 / 17.2; 20.5 / 21.8; and beyond: [12288 x 5120] (768) 1 14.6 / 14.0; 18.8 / 17.9, 2 14.5 / 17.2; 18.8 / 20.9,
// 4 14.8 / 22.4; 19.1 / 26.6, [10240 x 8192] (640) 4 18.4 / 25.0; 24.3 / 29.6, [24576 x 1536] (768) 1 11.6 / 9.6; 15.1 / 13.3, 4 12.0 / 14.8; 15.5 / 19.2.
constexpr int kQuantCost = 12, kQuantPerCu = 2;
constexpr int kQuantRows = 4, kQuantMaxK = 8192;  // QUANT: rows, and the values a lane holds of each (two vectors of 8)

// D: MFMA steps in flight; WPS: waves per SIMD the registers are cut for (4: two workgroups on a CU).
// QUANT (up to kQuantRows rows): the workgroup quantises the rows itself - every wave loads its part of K of each row,
// the waves exchange their maxima once, and the codes wait in LDS - with the arithmetic of quant_i8_rows_body, hence its
// bits; the weights are on their way meanwhile. A quantiser's launch less, 1 us of GPU time and 4 of the host's ([1 x 7168]
// x [4096 x 7168], weights in cache: 4.8 + 5.5 us -> 9.3). More rows cost more than the launch: 5 us per four.
template <int MF, int NF, int D, int WPS, bool QUANT = false>
__global__ __launch_bounds__(kDenseWaves* kWave, WPS) void dense_i8_kernel(const DenseParams p) {
  static_assert(!QUANT || MF == 1, "a few rows");
  constexpr int kFrags = MF * NF;
  __shared__ v4i red[kDenseWaves][kFrags][kWave];
  __shared__ uint32_t qmax[QUANT ? kQuantRows : 1][kDenseWaves];
  extern __shared__ __attribute__((aligned(16))) int8_t qrows[];  // QUANT: [rows][k + 16] codes
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int ksteps = p.k / 64;
  const int kb_begin = ksteps * wave / kDenseWaves, kb_end = ksteps * (wave + 1) / kDenseWaves;
  const int klen = kb_end - kb_begin;
  const int tile0 = blockIdx.y * p.tile_rows;
  const int tile_end = min(p.rows, tile0 + p.tile_rows);
  const int frag0 = blockIdx.x * NF;
  const int n_frags = p.n / 16;
  const int rot = p.rotate && klen > 1
                      ? static_cast<int>((((blockIdx.x * kDenseWaves + wave) * 2654435761u) >> 12) % static_cast<unsigned>(klen)) : 0;
  auto step_of = [&](int i) {
    const int s = i + rot;
    return static_cast<uint32_t>(kb_begin + (s >= klen ? s - klen : s));
  };

  // (fragments past the last channel and rows past the tile's end lie past their descriptor's end: they read zero)
  const uint32_t frag_bytes = static_cast<uint32_t>(ksteps) * 1024u;
  __amdgpu_buffer_rsrc_t wr[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    wr[f] = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.w + static_cast<size_t>(min(frag0 + f, n_frags - 1)) * frag_bytes), 0,
                                              frag0 + f < n_frags ? frag_bytes : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.a), 0, QUANT ? 0 : static_cast<uint32_t>(p.a_rows) * static_cast<uint32_t>(p.k), 0x00020000);
  uint32_t aoff[MF];
#pragma unroll
  for (int m = 0; m < MF; ++m) {
    const int r = tile0 + m * 16 + li;
    aoff[m] = r < tile_end ? static_cast<uint32_t>(p.src0 + r) * 64u + lg * 16u : 0xfffffff0u;
  }
  const uint32_t a_step = static_cast<uint32_t>(p.a_rows) * 64u;

  v4i wreg[D][NF], areg[QUANT ? 1 : D][MF];
  auto load_step = [&](int slot, int i) {
#pragma unroll
    for (int f = 0; f < NF; ++f) wreg[slot][f] = buffer_load16(wr[f], lane * 16, step_of(i) * 1024u);
    if constexpr (!QUANT) {
#pragma unroll
      for (int m = 0; m < MF; ++m) areg[slot][m] = buffer_load16(ar, aoff[m], step_of(i) * a_step);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < klen) load_step(d, d);

  // the scales of the fragments this wave finishes, on their way during the main loop
  constexpr int kOwn = (kFrags + kDenseWaves - 1) / kDenseWaves;
  float4 wm[kOwn];
  float am[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    const int f = wave + o * kDenseWaves;
    const int frag = frag0 + f % NF, r = tile0 + f / NF * 16 + li;
    wm[o] = f < kFrags && frag < n_frags ? *reinterpret_cast<const float4*>(p.w_max + frag * 16 + lg * 4) : make_float4(0, 0, 0, 0);
    am[o] = !QUANT && f < kFrags && r < tile_end ? p.a_max[p.src0 + r] : 0.0f;
  }

  const int pitch = p.k + 16;  // rows start 16 bytes further into the banks
  if constexpr (QUANT) {
    const bool f16 = p.f16 != 0;
    Pack8 v[kQuantRows][2];
    const int v0 = kb_begin * 8, nvec = klen * 8;  // this wave's vectors of 8 values of every row
#pragma unroll
    for (int r = 0; r < kQuantRows; ++r)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        v[r][i].v = make_uint4(0, 0, 0, 0);
        if (r < p.rows && lane + i * kWave < nvec)
          v[r][i].v = reinterpret_cast<const uint4*>(p.x + static_cast<size_t>(r) * p.ld_x)[v0 + lane + i * kWave];
      }
#pragma unroll
    for (int r = 0; r < kQuantRows; ++r) {
      if (r >= p.rows) break;
      const float m = fmaxf(amax8(v[r][0], f16), amax8(v[r][1], f16));
      const uint32_t bits = group_max_u32<kWave>(__builtin_bit_cast(uint32_t, m));  // (no negative numbers: ordered as their bits)
      if (lane == 0) qmax[r][wave] = bits;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kQuantRows; ++r) {
      if (r >= p.rows) break;
      uint32_t bits = qmax[r][0];
#pragma unroll
      for (int w = 1; w < kDenseWaves; ++w) bits = max(bits, qmax[r][w]);
      const float m = __builtin_bit_cast(float, bits);
      if (r == li) am[0] = m;
      const float inv = m > 0.0f ? 127.0f / m : 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (lane + i * kWave >= nvec) continue;
        *reinterpret_cast<uint2*>(&qrows[r * pitch + (v0 + lane + i * kWave) * 8]) = quant8_i8(v[r][i], inv, f16);
      }
    }
  }

  v4i acc[MF][NF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = (v4i){0, 0, 0, 0};
  // (rows a QUANT launch does not have repeat the last one: never stored)
  const int8_t* qp = &qrows[min(li, p.rows - 1) * pitch + lg * 16];
  for (int i0 = 0; i0 < klen; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (i0 + d < klen) {
#pragma unroll
        for (int m = 0; m < MF; ++m) {
          const v4i av = QUANT ? *reinterpret_cast<const v4i*>(qp + step_of(i0 + d) * 64) : areg[QUANT ? 0 : d][m];
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[m][f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[d][f], av, acc[m][f], 0, 0, 0);
        }
        if (i0 + d + D < klen) load_step(d, i0 + d + D);
      }
    }
  }

#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) red[wave][m * NF + f][lane] = acc[m][f];
  __syncthreads();
#pragma unroll
  for (int o = 0; o < kOwn; ++o) {
    const int f = wave + o * kDenseWaves;
    const int frag = frag0 + f % NF, r = tile0 + f / NF * 16 + li;
    if (f >= kFrags || frag >= n_frags || r >= tile_end) continue;
    v4i sum = red[0][f][lane];
#pragma unroll
    for (int w = 1; w < kDenseWaves; ++w) sum += red[w][f][lane];
    const float sa = am[o] / 127.0f;
    const float sw[4] = {wm[o].x / 127.0f, wm[o].y / 127.0f, wm[o].z / 127.0f, wm[o].w / 127.0f};
    uint16_t out[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = f32_to_act((static_cast<float>(sum[q]) * sa) * sw[q], p.f16 != 0);
    const size_t row = p.row0 + r;
    const int c = frag * 16 + lg * 4;
    if (p.acc_out) *reinterpret_cast<v4i*>(p.acc_out + row * p.n + c) = sum;
    *reinterpret_cast<uint2*>(p.y + row * p.ldy + c) =
        make_uint2(out[0] | (static_cast<uint32_t>(out[1]) << 16), out[2] | (static_cast<uint32_t>(out[3]) << 16));
  }
}

template <int MF, int NF, int D, int WPS, bool QUANT = false>
int launch_dense(DenseParams p, hipStream_t s) {
  const int tiles = ceil_div(p.rows, 16 * MF);
  p.tile_rows = ceil_div(p.rows, tiles);
  if (tracing_kernels())
    note_kernel("dense_i8_kernel<%d x %d tile, K split %d, %d steps in flight%s>", 16 * MF, 16 * NF, kDenseWaves, D,
                QUANT ? ", quantises its rows itself" : "");
  const size_t lds = QUANT ? static_cast<size_t>(p.rows) * (p.k + 16) : 0;
  hipLaunchKernelGGL((dense_i8_kernel<MF, NF, D, WPS, QUANT>), dim3(ceil_div(p.n, 16 * NF), tiles), dim3(kDenseWaves * kWave), lds, s, p);
  return check_launch("kmoe_grouped_gemm_i8 (dense)");
}

// Fragments (16 channels of k codes) begin a multiple of 32 KB apart where this holds, and waves in step ask the same
// channels of memory: each starts its part of K at a step of its own (whole-number sums: same bits). GEMM alone, us, all
// waves at the first step / rotated, weights cold: [7168 x 2048] 24 rows 5.8 / 5.5, 33 7.5 / 6.6, 100 8.4 / 8.1, 128 9.3 /
// 8.7; [4096 x 2048] 200 9.4 / 8.6; [12288 x 2048] 64 11.9 / 10.9; [6144 x 6144] 80 16.6 / 16.1; 1 to 16 rows, k = 10240 and
// weights in cache level. Other k gain a little or lose a little: [4096 x 2560] 33 rows 5.0 / 4.8, [4096 x 1024] 100 4.7 /
// 4.8, [4096 x 7168] 100 11.2 / 11.4.
bool rotates(int k) { return k % 2048 == 0; }

// The tiles, and what a launch on one costs: rounds of workgroups over the CUs times the KB a workgroup fetches per K step
// (MF + NF). The cheapest tile, the smaller of equals, is within 0.2 % of the fastest on average and 7 % at worst over
// eight matrices ([4096 x 7168], [7168 x 2048], [8192 x 8192], [12288 x 5120], [24576 x 1536], [1536 x 7168], [2048 x 2048],
// [576 x 7168]) and 1 to 512 rows each, weights cold. Examples, GEMM alone, us, streaming kernel or tile kernel whichever
// was taken before -> now: [4096 x 7168] 1 row 11.3 -> 7.7, 32 12.7 -> 9.9, 64 15.7 -> 11.5, 100 17.9 -> 13.7, 256 26.3 -> 19.2;
// [7168 x 2048] 1 row 5.8 -> 4.8, 64 8.6 -> 6.8, 128 8.7 -> 8.3; [8192 x 8192] 64 rows 25.0 -> 19.0; [1536 x 7168] 128 rows
// 11.0 -> 7.9.
struct DenseShape {
  int mf, nf;
};
constexpr DenseShape kDenseShapes[] = {{1, 1}, {1, 2}, {2, 2}, {4, 2}, {4, 4}};

int dense_cost(int n, int rows, int n_cu, int* shape) {
  int best = 1 << 30;
  for (int i = 0; i < 5; ++i) {
    const DenseShape t = kDenseShapes[i];
    const long long groups = static_cast<long long>(ceil_div(n, 16 * t.nf)) * ceil_div(rows, 16 * t.mf);
    const long long cost = (groups + n_cu - 1) / n_cu * (t.mf + t.nf);
    if (cost < best) {
      best = static_cast<int>(cost);
      *shape = i;
    }
  }
  return best;
}

int launch_shape(const DenseParams& p, int shape, hipStream_t s) {
  switch (shape) {
    case 0: return launch_dense<1, 1, 8, 4>(p, s);
    case 1: return launch_dense<1, 2, 8, 4>(p, s);
    case 2: return launch_dense<2, 2, 5, 4>(p, s);
    case 3: return launch_dense<4, 2, 3, 4>(p, s);
    default: return launch_dense<4, 4, 3, 2>(p, s);
  }
}

}  // namespace

// (up to 16 rows there is always one row tile, whatever the channels; the tile kernel, which reads the weights once per
// 32 to 192 rows, is level or ahead where the launch costs 16 and more: [4096 x 7168] 384 rows 30.1 / 31.6 us, [12288 x
// 5120] 96 rows 24.7 / 27.5, [24576 x 1536] 48 rows 11.7 / 12.0; [1536 x 7168] 512 rows, cost 8: 19.0 / 15.1)
constexpr int kDenseCost = 15, kDenseMaxRows = 512;

bool dense_gemm_i8_reaches(int a_rows, int k) { return static_cast<int64_t>(a_rows) * k < 0xfff00000ll; }

int dense_gemm_i8(const kmoe_gemm_i8_args* a, hipStream_t s) {
  int n_cu = 0, shape = 0;
  if (int rc = compute_units(&n_cu)) return rc;
  DenseParams p = {};
  p.a = a->a;
  p.a_rows = a->a_rows;
  p.src0 = a->tail_src0;
  p.a_max = a->a_max;
  p.w = a->w_tail;
  p.w_max = a->w_max_tail;
  p.n = a->n;
  p.k = a->k;
  p.rows = a->tail_rows;
  p.row0 = a->tail_row0;
  p.y = a->y;
  p.ldy = a->ldy;
  p.acc_out = a->acc_out;
  p.f16 = a->act_dtype == KMOE_DT_F16;
  p.rotate = rotates(a->k);
  dense_cost(a->n, a->tail_rows, n_cu, &shape);
  return launch_shape(p, shape, s);
}

}  // namespace kmoe

using namespace kmoe;

extern "C" int kmoe_linear_i8_split_rows(int n, int k) {
  int n_cu = 0, shape = 0, rows = 16;
  if (n < 16 || k < 64 || n % 16 != 0 || k % 64 != 0 || k > 65536) return 0;
  if (compute_units(&n_cu)) return rows;
  while (rows < kDenseMaxRows && dense_cost(n, rows + 1, n_cu, &shape) <= kDenseCost) ++rows;  // (the cost grows with the rows)
  return rows;
}

extern "C" size_t kmoe_linear_i8_workspace_bytes(int rows, int k) {
  return align_up(static_cast<size_t>(rows) * k, 256) + static_cast<size_t>(rows) * 4;
}

extern "C" int kmoe_linear_i8(const kmoe_linear_i8_args* a, kmoe_stream_t stream) {
  KMOE_REQUIRE(a, KMOE_ERR_NULL, "linear_i8: args is NULL");
  KMOE_REQUIRE(a->x && a->w && a->w_max && a->y && a->scratch, KMOE_ERR_NULL, "linear_i8: NULL pointer");
  KMOE_REQUIRE(a->rows >= 0 && a->n >= 16 && a->k >= 16 && a->n % 16 == 0 && a->k % 16 == 0 && a->k <= 65536, KMOE_ERR_SHAPE,
               "linear_i8: rows=%d n=%d k=%d", a->rows, a->n, a->k);
  KMOE_REQUIRE(a->scratch_bytes >= kmoe_linear_i8_workspace_bytes(a->rows, a->k) && (reinterpret_cast<uintptr_t>(a->scratch) & 255) == 0,
               KMOE_ERR_WORKSPACE, "linear_i8: scratch of %zu bytes, need %zu, 256-byte aligned", a->scratch_bytes,
               kmoe_linear_i8_workspace_bytes(a->rows, a->k));
  if (a->rows == 0) return KMOE_OK;
  kmoe_gemm_i8_args g = {};
  g.a = static_cast<const int8_t*>(a->scratch);
  float* x_max = reinterpret_cast<float*>(static_cast<char*>(a->scratch) + align_up(static_cast<size_t>(a->rows) * a->k, 256));
  g.a_max = x_max;
  g.lda = a->k;
  g.src_div = 1;
  g.w = a->w;
  g.w_max = a->w_max;
  g.E = 1;
  g.n = a->n;
  g.k = a->k;
  g.y = a->y;
  g.ldy = a->ldy;
  g.w_layout = a->w_layout;
  g.act_dtype = a->act_dtype;
  if (a->lod) {  // rows enough for the tile kernel, or row-major weights: row-major codes, one expert
    if (int rc = kmoe_quant_i8_rows_dt(a->x, a->ld_x, a->rows, a->k, static_cast<int8_t*>(a->scratch), a->k, x_max, a->act_dtype, stream)) return rc;
    g.lod = a->lod;
    g.rows = a->rows;
    return kmoe_grouped_gemm_i8(&g, stream);
  }
  KMOE_REQUIRE(a->w_layout == KMOE_W_TILED && a->k % 64 == 0, KMOE_ERR_UNSUPPORTED, "linear_i8: without lod the weights must be tiled");
  KMOE_REQUIRE(a->act_dtype == KMOE_DT_BF16 || a->act_dtype == KMOE_DT_F16, KMOE_ERR_UNSUPPORTED, "linear_i8: act_dtype=%d unknown", a->act_dtype);
  KMOE_REQUIRE(a->ld_x % 8 == 0 && a->ld_x >= a->k && a->ldy % 4 == 0 && a->ldy >= a->n, KMOE_ERR_SHAPE, "linear_i8: strides %lld/%lld",
               static_cast<long long>(a->ld_x), static_cast<long long>(a->ldy));
  auto aligned = [](const void* q, uintptr_t to) { return (reinterpret_cast<uintptr_t>(q) & (to - 1)) == 0; };
  KMOE_REQUIRE(aligned(a->w, 16) && aligned(a->w_max, 16) && aligned(a->y, 8), KMOE_ERR_SHAPE, "linear_i8: misaligned tensor pointer");
  if (a->rows <= kQuantRows && a->k <= kQuantMaxK && aligned(a->x, 16)) {
    int n_cu = 0, shape = 0;
    if (int rc = compute_units(&n_cu)) return rc;
    const int cost = dense_cost(a->n, a->rows, n_cu, &shape);
    if (cost <= kQuantCost && (a->rows == 1 || ceil_div(a->n, 16 * kDenseShapes[shape].nf) <= kQuantPerCu * n_cu)) {
      DenseParams p = {};
      p.x = a->x;
      p.ld_x = a->ld_x;
      p.w = a->w;
      p.w_max = a->w_max;
      p.n = a->n;
      p.k = a->k;
      p.rows = a->rows;
      p.y = a->y;
      p.ldy = a->ldy;
      p.f16 = a->act_dtype == KMOE_DT_F16;
      p.rotate = rotates(a->k);
      return shape == 0 ? launch_dense<1, 1, 8, 4, true>(p, as_stream(stream)) : launch_dense<1, 2, 5, 4, true>(p, as_stream(stream));
    }
  }
  KMOE_REQUIRE(dense_gemm_i8_reaches(a->rows, a->k), KMOE_ERR_SHAPE, "linear_i8: %d rows of %d codes need 32-bit offsets without lod", a->rows, a->k);
  if (int rc = kmoe_quant_i8_rows_chunked_dt(a->x, a->ld_x, a->rows, a->k, static_cast<int8_t*>(a->scratch), x_max, a->act_dtype, stream)) return rc;
  g.a_layout = KMOE_A_CHUNKED;
  g.a_rows = a->rows;
  g.w_tail = a->w;
  g.w_max_tail = a->w_max;
  g.tail_rows = a->rows;
  return dense_gemm_i8(&g, as_stream(stream));
}
