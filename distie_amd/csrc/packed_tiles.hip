// Products of many rows on packed weight copies: y[M, N] = x[M, K] W[N, K]^T for bfloat16 x and the copies of packed.h.
//
// The copies hold W as tiles of 16 rows x 32 k in the matrix cores' lane order, so a wave reads its operand of W
// straight into registers, 1 KB of consecutive bytes an instruction, and only x goes through LDS. A workgroup of four
// waves owns a tile of 16 MB rows of x and 64 NB rows of W (16 NB a wave) and one slice of K; a stage is 64 k.
//
// What bounds it. Small tiles (DEPTH 4): the workgroups that share rows of W ask for the same lines at the same time, so
// what is under way from memory is a fraction of what the compute units wait for, and a stage ahead is not enough: four
// stages of x and W are under way in registers (waited for by count), x goes from there into LDS (down of the 1.5B shape,
// [301, 8960] x [1536, 8960]: 20.2 -> 18.1 us; [64, 8960]: 11.5 -> 9.1). Large tiles (DEPTH 2): the matrix cores, which
// the whole chip's power holds at two thirds of their nominal rate, and the L2 (12 to 17 TB/s reach the compute units):
// one stage ahead, x without a stop in registers, which the sums need. [2025, 3584] x [37888, 3584] runs at 1,063 TFLOP/s
// (517 us; gated 957, 573 us in either large tile, where the library and the activation's kernel take 567), the same loop
// without any loads at 1,460. Three parts of LDS there, 32 x 32 products, or touching the lines of later stages for the L2
// changed nothing or lost up to a fifth.

#include "common.h"
#include "lds_load.h"
#include "packed.h"
#include <algorithm>

namespace {

constexpr int PT_K = 64;              // k of a stage

// As `load_to_lds`, in its place among the reads and writes of memory around it (they stand in the order written).
__device__ __forceinline__ void stage_to_lds(const bf16_t* from, bf16_t* to) {
  asm volatile("" ::: "memory");
  load_to_lds(from, lds_place(to));
  asm volatile("" ::: "memory");
}

struct TilesPlace {
  int row_blocks;               // blocks of 16 rows of the packed copy
  int m_tiles, n_tiles, slices;
  int stages;                   // of a slice
};

// MODE: PK_PLAIN, PK_GATED, PK_ROTARY. K a multiple of PT_K.
template <int MB, int NB, int DEPTH, int MODE, typename Y>
__global__ __launch_bounds__(256, 2) void packed_tiles_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              const float* __restrict__ bias, Y* __restrict__ y, int M, int N,
                                                              int K, TilesPlace at, RotaryOut rotary) {
  constexpr int ROWS = 16 * MB;
  constexpr int PARTS = MB / 2;       // pieces of 16 bytes of x's stage that a thread brings
  __shared__ __attribute__((aligned(16))) bf16_t xs[2][ROWS * PT_K];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
  // Workgroup i runs on die i % 8: every die gets a run of neighbouring tiles, the rows of x fastest, so that the
  // workgroups at work on a die read the same few parts of W and of x through its L2.
  const int tiles = at.m_tiles * at.n_tiles;
  const int place = static_cast<int>(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (place >= tiles * at.slices) return;
  const int slice = place / tiles, n_tile = place % tiles / at.m_tiles, m_tile = place % at.m_tiles;
  const int m0 = m_tile * ROWS;
  const int k_tiles = K / 32;
  const int s_begin = slice * at.stages;
  const int stages = min(K / PT_K - s_begin, at.stages);
  const int block0 = (n_tile * 4 + wave) * NB;
  const bf16_t* wp[NB];               // blocks beyond the last are read from it and dropped
#pragma unroll
  for (int n = 0; n < NB; ++n)
    wp[n] = w + (static_cast<int64_t>(min(block0 + n, at.row_blocks - 1)) * k_tiles + 2 * s_begin) * PK_TILE + lane * 8;
  // A row of x's stage is eight pieces of 16 bytes; eight neighbouring lanes bring a row (128 bytes in one run). Piece p
  // lies at place p ^ (row / 2 % 8), so that the sixteen rows a product reads at once spread over all banks.
  const int row = tid / 8, piece = (tid % 8) ^ ((row >> 1) & 7);
  const bf16_t* xp[PARTS];
#pragma unroll
  for (int p = 0; p < PARTS; ++p)
    xp[p] = x + static_cast<int64_t>(min(m0 + 32 * p + row, M - 1)) * K + PT_K * s_begin + 8 * piece;
  floatx4 acc[NB][MB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[n][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[DEPTH][NB][2];
  auto fetch_w = [&](int stage, int slot) {
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        a[slot][n][j] = *reinterpret_cast<const bf16x8*>(wp[n] + static_cast<int64_t>(2 * stage + j) * PK_TILE);
  };
  auto multiply = [&](int half, int slot) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bf16_t* from = &xs[half][r * PT_K + 8 * ((4 * j + g) ^ (r >> 1))];
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        const bf16x8 xb = *reinterpret_cast<const bf16x8*>(from + b * 16 * PT_K);
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[n][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[slot][n][j], xb, acc[n][b], 0, 0, 0);
      }
    }
  };
  if constexpr (DEPTH == 2) {
    auto fetch = [&](int stage, int half) {
#pragma unroll
      for (int p = 0; p < PARTS; ++p) stage_to_lds(xp[p] + PT_K * stage, &xs[half][(32 * p + 8 * wave) * PT_K]);
      fetch_w(stage, half);
      __builtin_amdgcn_sched_barrier(0);         // (else the compiler asks late for what the next stage needs)
    };
    fetch(0, 0);
    int s = 0;
    for (; s + 2 <= stages; s += 2) {
      lds_arrived<0>();
      fetch(s + 1, 1);
      multiply(0, 0);
      lds_arrived<0>();
      fetch(min(s + 2, stages - 1), 0);          // (past the last stage: the last once more, not used)
      multiply(1, 1);
    }
    lds_arrived<0>();                               // nothing is under way when the workgroup ends
    if (s < stages) multiply(0, 0);
  } else {
    bf16x8 xr[DEPTH][PARTS];
    auto fetch = [&](int stage, int slot) {
      const int at_stage = min(stage, stages - 1);
      fetch_w(at_stage, slot);
#pragma unroll
      for (int p = 0; p < PARTS; ++p) xr[slot][p] = *reinterpret_cast<const bf16x8*>(xp[p] + PT_K * at_stage);
    };
    auto step = [&](int slot) {
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
        *reinterpret_cast<bf16x8*>(&xs[slot % 2][(32 * p + row) * PT_K + 8 * (tid % 8)]) = xr[slot][p];
      __syncthreads();
      multiply(slot % 2, slot);
    };
#pragma unroll
    for (int slot = 0; slot < DEPTH; ++slot) fetch(slot, slot);
    int s = 0;
    for (; s + 2 * DEPTH <= stages; s += DEPTH) {
#pragma unroll
      for (int slot = 0; slot < DEPTH; ++slot) {
        step(slot);
        fetch(s + slot + DEPTH, slot);
      }
    }
#pragma unroll
    for (int q = 0; q < 2 * DEPTH - 1; ++q) {
      if (s + q < stages) {
        step(q % DEPTH);
        if (q < DEPTH && s + q + DEPTH < stages) fetch(s + q + DEPTH, q % DEPTH);
      }
    }
  }

  // acc[n][b][i]: row 4 g + i of block block0 + n, row 16 b + r of x's tile
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int block = block0 + n;                // (the same in all lanes of a wave)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      if (block >= at.row_blocks) continue;
      const int m = m0 + 16 * b + r;
      float v[4] = {acc[n][b][0], acc[n][b][1], acc[n][b][2], acc[n][b][3]};
      if constexpr (MODE == PK_GATED) {
        float up[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(v[i], 32, 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gated_value(v[i], up[i], rotary.act, rotary.limit, rotary.slope, rotary.up_shift);
        if (g < 2 && m < M) store_four(y + static_cast<int64_t>(m) * (N / 2), 8 * block + 4 * g, N / 2, v);
      } else if constexpr (MODE == PK_ROTARY) {
        store_rotary(v, m, m < M, g, block, bias, y, N, rotary);
      } else {
        const int n0 = 16 * block + 4 * g;
        if (bias != nullptr && slice == 0) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] += n0 + i < N ? bias[n0 + i] : 0.f;
        }
        if (m < M) store_four(y + static_cast<int64_t>(slice) * M * N + static_cast<int64_t>(m) * N, n0, N, v);
      }
    }
  }
}

// The tiles there are, and what a workgroup of one takes: a start, and for every stage (and `more` of them to begin and
// end) alone_us with a compute unit to itself (its trip to the L2) up to full_us with all `residents` on it.
struct TileCost {
  float start_us, alone_us, full_us, more;
};
struct TileShape {
  int mb, nb;
  int residents;                // workgroups of it that share a compute unit (their registers decide)
  TileCost plain, gated;        // (the weights of gated products are the large ones, which all come from memory)
};
constexpr TileShape SHAPES[] = {
    {4, 1, 4, {3.0f, 0.21f, 0.79f, 3.5f}, {3.3f, 0.39f, 0.96f, 0.f}},
    {4, 2, 3, {3.2f, 0.29f, 0.88f, 4.6f}, {5.7f, 0.53f, 1.13f, 0.f}},
    {6, 2, 2, {2.9f, 0.41f, 0.76f, 5.8f}, {7.5f, 0.54f, 0.90f, 3.7f}},
    {8, 2, 3, {0.3f, 0.68f, 1.34f, 8.1f}, {5.6f, 0.86f, 1.46f, 5.3f}},
    {8, 4, 2, {0.6f, 0.95f, 1.60f, 8.2f}, {3.4f, 1.45f, 1.78f, 11.8f}}};
constexpr int SHAPE_COUNT = static_cast<int>(sizeof(SHAPES) / sizeof(SHAPES[0]));
constexpr int LARGE_TILES_FROM = 193;     // rows of x from which the two largest are considered: below, most of a tile is padding

struct TilesPlan {
  int shape, slices;
  float us;
};

// How a product is cut: the shape and the number of slices for which a simple count comes out lowest: whole rounds of
// workgroups on the compute units, each as long as its stages, no faster than memory brings W, and what the reader of
// several float32 slices has to move beside one bfloat16 result. The numbers above are a least-squares fit to 4,600 timings
// (17 to 2,048 rows, weights of 1024 x 1024 to 37888 x 3584, each read from memory; the fit is off by 5 to 10 %). What the
// count chooses takes 1.3 % more than the best of them on average, 21 % at worst. `cut_us`: what a cut costs the caller
// beyond that (a kernel that adds the slices up).
TilesPlan plan_tiles(int M, int N, int K, int row_blocks, bool gated, bool may_cut, float cut_us) {
  TilesPlan best = {-1, 0, 0.f};
  const int all = K / PT_K;
  const float memory_us = static_cast<float>(row_blocks) * K * 32.f / 4.6e6f;
  for (int i = 0; i < (M < LARGE_TILES_FROM ? 3 : SHAPE_COUNT); ++i) {
    const TileShape& s = SHAPES[i];
    const int tiles = ((M + 16 * s.mb - 1) / (16 * s.mb)) * ((row_blocks + 4 * s.nb - 1) / (4 * s.nb));
    for (int cut = 1; cut <= 12; ++cut) {
      if (cut > 1 && (!may_cut || all / cut < 4)) break;
      const int stages = (all + cut - 1) / cut;
      if ((all + stages - 1) / stages != cut) continue;
      const TileCost& c = gated ? s.gated : s.plain;
      const auto stage_us = [&](int r) { return c.alone_us + (c.full_us - c.alone_us) * (r - 1) / (s.residents - 1); };
      const int per_unit = (tiles * cut + 255) / 256, rest = per_unit % s.residents;
      float us = (per_unit / s.residents) * stage_us(s.residents) + (rest > 0 ? stage_us(rest) : 0.f);
      us = c.start_us + std::max(us * (stages + c.more), memory_us);
      if (cut > 1) us += (4.f * cut - 2.f) * M * N / 4.5e6f + cut_us;
      if (best.shape < 0 || us < best.us) best = {i, cut, us};
    }
  }
  return best;
}

template <int MODE, typename Y>
int launch_tiles(const bf16_t* x, const bf16_t* w, const float* bias, Y* y, int M, int N, int K, int row_blocks, int shape,
                 int slices, const RotaryOut& rotary, hipStream_t stream) {
  const TileShape s = SHAPES[shape];
  const int all = K / PT_K;
  TilesPlace at = {row_blocks, (M + 16 * s.mb - 1) / (16 * s.mb), (row_blocks + 4 * s.nb - 1) / (4 * s.nb), slices,
                   (all + slices - 1) / slices};
  if ((all + at.stages - 1) / at.stages != slices) return DISTIE_BAD_ARGUMENT;
  const int64_t work = static_cast<int64_t>(at.m_tiles) * at.n_tiles * slices;
  if (work > (1 << 30)) return DISTIE_BAD_ARGUMENT;
  const unsigned grid = static_cast<unsigned>((work + 7) / 8 * 8);
#define TILES(MB, NB, DEPTH) packed_tiles_kernel<MB, NB, DEPTH, MODE, Y><<<grid, 256, 0, stream>>>(x, w, bias, y, M, N, K, at, rotary)
  switch (shape) {
    case 0: TILES(4, 1, 4); break;
    case 1: TILES(4, 2, 4); break;
    case 2: TILES(6, 2, 4); break;
    case 3: TILES(8, 2, 2); break;
    default: TILES(8, 4, 2); break;
  }
#undef TILES
  return launch_status();
}

int row_blocks_of(int N, bool gated) { return gated ? (N / 2 + 7) / 8 : (N + 15) / 16; }

}  // namespace

// How the kernels of this file cut a product; 0 if they do not take it. gated: the copy's rows are gate and up in turn;
// may_cut: the caller takes float32 slices, at cut_us more. *shape and *slices go to the launch as they are; *workgroups: how
// many it will have.
extern "C" int distie_packed_tiles_plan(int M, int N, int K, int gated, int may_cut, float cut_us, int* shape, int* slices,
                                        int* workgroups) {
  if (M < 1 || N < 1 || K < 2 * PT_K || K % PT_K != 0 || (gated && N % 2 != 0)) return 0;
  const TilesPlan plan = plan_tiles(M, N, K, row_blocks_of(N, gated != 0), gated != 0, may_cut != 0 && !gated, cut_us);
  const TileShape& s = SHAPES[plan.shape];
  const int64_t blocks = row_blocks_of(N, gated != 0);
  const int64_t all = (static_cast<int64_t>(M) + 16 * s.mb - 1) / (16 * s.mb) * ((blocks + 4 * s.nb - 1) / (4 * s.nb)) * plan.slices;
  *shape = plan.shape, *slices = plan.slices, *workgroups = static_cast<int>(std::min<int64_t>(all, 1 << 30));
  return 1;
}

// y: [M, N] of y_dtype (gated: [M, N / 2] in bfloat16), or with slices > 1 float32 [slices, M, N], to be added in order by
// whoever reads it, the bias in the first.
extern "C" int distie_packed_tiles_bf16(const void* x, const void* w_packed, const float* bias, void* y, int y_dtype, int M,
                                        int N, int K, int gated, int shape, int slices, float limit, float slope, float up_shift,
                                        hipStream_t stream) {
  if (M <= 0) return 0;
  const int act = gated >> 8;           // the activation on the gate, above the low eight bits
  gated &= 0xff;
  if (N < 1 || K < 2 * PT_K || K % PT_K != 0 || shape < 0 || shape >= SHAPE_COUNT ||
      slices < 1 || gated > 1 || (gated && (N % 2 != 0 || slices != 1 || y_dtype != DISTIE_BF16 || bias != nullptr)) || act < 0 ||
      act > 5 || (act == 5 && !(limit > 0.f)) || (slices > 1 && y_dtype != DISTIE_F32))
    return DISTIE_BAD_ARGUMENT;
  RotaryOut out = {};
  out.act = act, out.limit = limit, out.slope = slope, out.up_shift = up_shift;
  const bf16_t* xb = static_cast<const bf16_t*>(x);
  const bf16_t* wb = static_cast<const bf16_t*>(w_packed);
  const int blocks = row_blocks_of(N, gated != 0);
  if (gated) return launch_tiles<PK_GATED, bf16_t>(xb, wb, nullptr, static_cast<bf16_t*>(y), M, N, K, blocks, shape, 1, out, stream);
  DISTIE_DISPATCH(y_dtype, Y, return (launch_tiles<PK_PLAIN, Y>(xb, wb, bias, static_cast<Y*>(y), M, N, K, blocks, shape, slices,
                                                                out, stream)));
  return DISTIE_BAD_ARGUMENT;
}

// The stacked q/k/v product with rotation and cache write in its epilogue, as distie_gemm_packed_rotary_bf16.
extern "C" int distie_packed_tiles_rotary_bf16(const void* x, const void* w_packed, const float* bias, void* y,
                                               const void* table, const int32_t* slots, void* k_cache, void* v_cache, int M,
                                               int K, int heads, int kv_heads, int dim, int block_size, int write, int shape,
                                               hipStream_t stream) {
  if (M <= 0) return 0;
  if (K < 2 * PT_K || K % PT_K != 0 || heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 != 0 || block_size < 1 ||
      shape < 0 || shape >= SHAPE_COUNT || table == nullptr ||
      (write && (slots == nullptr || k_cache == nullptr || v_cache == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const int N = (heads + 2 * kv_heads) * dim;
  const RotaryOut rotary = {static_cast<const float2*>(table), slots, static_cast<bf16_t*>(k_cache),
                            static_cast<bf16_t*>(v_cache), heads, kv_heads, dim, block_size, write};
  return launch_tiles<PK_ROTARY, bf16_t>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w_packed), bias,
                                         static_cast<bf16_t*>(y), M, N, K, N / 16, shape, 1, rotary, stream);
}
