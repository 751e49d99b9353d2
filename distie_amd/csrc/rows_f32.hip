// The true 32-bit path's products of few rows of x on the matrix cores: y[M, N] = x[M, K] W[N, K]^T, float32 operands,
// products and sums (v_mfma_f32_16x16x4_f32: no mode of reduced precision), W in the checkpoint's layout.
//
// A wave owns 16 rows of W (the A operand) and streams its share of K; up to 32 rows of x are the B operand, 16 a block.
// A lane's sixteen bytes of a row of W or x hold four k, which four products take one after the other: the summed index
// runs in the lanes' order (lane 16 g + r: row r, k 4 g .. 4 g + 3 of every 16), the same for both. Which rows a wave
// owns is free, as W is not packed: gate rows beside their up rows, or the partners of a rotation, so that activation,
// rotation and cache write happen in the epilogue as in the bfloat16 products.
//
// What bounds it. Few rows: W from memory, large weights at 3.3 to 4.5 TB/s (a read of weights alone reaches 6.4: a wave's loads
// touch 64 bytes of each of 16 rows); 32 rows: the matrix instructions and the loads of x beside them, at 2.4 TB/s of W; q/k/v,
// whose weights are small: its launch and one wave's chain of trips to memory. Large weights go through LDS in whole lines instead
// (`rows_f32_tiles_kernel`, and where it is taken, `rows_tiles`), x with them: 4.1 TB/s at 8 and at 16 rows, 5.5 of the 7B shape's gate+up.
// The kernel on registers, 1.5B shape, every weight from memory, us and TB/s of
// W at 1, 8, 32 rows, behind the slash us of the kernel on the vector ALU (gemv_rows) with what stands behind it: gate+up with
// activation 24.7 (4.5), 27.9 (4.0), 45.5 (2.4) / 27.4, 37.6, 82.2; down in 8 slices 16.1 (3.4), 16.8 (3.3), 22.5 (2.5) / 15.7, 21.7,
// 37.8; q/k/v with rotation and cache write 7.7 (1.6), 8.8 (1.4), 13.1 (1.0) / 11.2, 13.8, 23.6. With more than 32 rows the
// sums' chains no longer fit the registers at the precision of the vector ALU's kernel.

#include "common.h"
#include "lds_load.h"
#include "packed.h"
#include <algorithm>

namespace {

constexpr int RF_STEP = 64;           // k of a step: four loads of 16 bytes a lane and operand

struct RowsShare {
  const float* w;                     // the lane's row of W
  const float* x[2];                  // and of x, a block of 16 rows each
};

// COUNT steps, every load issued before the first product. Their products go into CHAINS sums that start at zero, which
// are added up in pairs and then to the total: one chain over the whole K rounds five times as far from the sum in 64
// bits (5e-7 of it at K = 1,536; the vector ALU's kernel, whose lanes keep sums of their own, 1.1e-7).
template <int MB, int COUNT>
__device__ __forceinline__ void rows_steps(const RowsShare& at, int begin, int steps, int& step, floatx4 (&total)[MB]) {
  constexpr int CHAINS = 16 / MB;
  floatx4 a[COUNT][4], b[COUNT][MB][4];
#pragma unroll
  for (int u = 0; u < COUNT; ++u) {
    const int k = RF_STEP * (begin + step);
    step = step + 1 == steps ? 0 : step + 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[u][j] = *reinterpret_cast<const floatx4*>(at.w + k + 16 * j);
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) b[u][m][j] = *reinterpret_cast<const floatx4*>(at.x[m] + k + 16 * j);
  }
  __builtin_amdgcn_sched_barrier(0);           // (left alone the compiler asks for each piece shortly before its use)
  floatx4 acc[CHAINS][MB];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[c][m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < COUNT; ++u)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          floatx4& c = acc[(4 * j + e) % CHAINS][m];
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][j][e], b[u][m][j][e], c, 0, 0, 0);
        }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
#pragma unroll
    for (int half = CHAINS / 2; half >= 1; half /= 2)
#pragma unroll
      for (int c = 0; c < half; ++c) acc[c][m] += acc[c + half][m];
    total[m] += acc[0][m];
  }
}

struct FourSums {
  float v[4];
};

// The end of a product: sums.v[i] is row 4 g + i of the block for row at_row of x (every lane of the wave has to come here).
template <int MODE>
__device__ __forceinline__ void rows_f32_store(FourSums sums, int block, int at_row, int g, const float* bias, float* y, int M, int N,
                                               const RotaryOut& rotary) {
  float (&v)[4] = sums.v;
  if constexpr (MODE == PK_GATED) {
    const int half = N / 2;
    float up[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(v[i], 32, 64);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gated_value(v[i], up[i], rotary.act, rotary.limit, rotary.slope, rotary.up_shift);
    if (g < 2 && at_row < M) store_four(y + static_cast<int64_t>(at_row) * half, 8 * block + 4 * g, half, v);
  } else if constexpr (MODE == PK_ROTARY) {
    store_rotary(v, at_row, at_row < M, g, block, bias, y, N, rotary);
  } else {
    const int n0 = 16 * block + 4 * g;
    if (bias != nullptr && blockIdx.y == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += n0 + i < N ? bias[n0 + i] : 0.f;
    }
    if (at_row < M) store_four(y + (static_cast<int64_t>(blockIdx.y) * M + at_row) * N, n0, N, v);
  }
}

// blockIdx.x: block of 16 rows; blockIdx.y: slice of K (plain products only; slices side by side in y, bias on the
// first). The waves of a workgroup share the slice's steps and add their sums through LDS; the first one writes.
template <int MB, int MODE, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void rows_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                              int K, int steps_per_slice, RotaryOut rotary) {
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, r = lane % 16, g = lane / 16;
  const int block = blockIdx.x;
  int64_t row;
  if constexpr (MODE == PK_GATED) {
    const int half = N / 2, j = min(8 * block + r % 8, half - 1);        // rows beyond the last: results dropped
    row = r < 8 ? j : half + j;
  } else if constexpr (MODE == PK_ROTARY) {
    row = rotary_column(block, r / 4, rotary.heads + rotary.kv_heads, rotary.dim) + r % 4;
  } else {
    row = min(16 * block + r, N - 1);
  }
  RowsShare at;
  at.w = w + row * K + 4 * g;
#pragma unroll
  for (int m = 0; m < 2; ++m) at.x[m] = x + static_cast<int64_t>(min(16 * m + r, M - 1)) * K + 4 * g;
  const int all = K / RF_STEP;
  const int s_begin = blockIdx.y * steps_per_slice, s_end = min(all, s_begin + steps_per_slice);
  const int share = (s_end - s_begin + WAVES - 1) / WAVES;
  const int begin = min(s_end, s_begin + wave * share), steps = min(s_end, begin + share) - begin;
  floatx4 acc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
  // workgroups begin at different steps and wrap around, so that they do not pull on the same memory channels at once
  int step = steps > 0 ? static_cast<int>((blockIdx.x + wave) % steps) : 0;
  constexpr int UN = MB == 1 && WAVES == 1 ? 4 : 2;      // (gate+up at 8 rows, four waves: two 29.8 us, four 31.6)
  int s = 0;
  for (; s + UN <= steps; s += UN) rows_steps<MB, UN>(at, begin, steps, step, acc);
  if constexpr (UN > 2) {
    if (steps - s >= 2) {
      rows_steps<MB, 2>(at, begin, steps, step, acc);
      s += 2;
    }
  }
  if (s < steps) rows_steps<MB, 1>(at, begin, steps, step, acc);

  if constexpr (WAVES > 1) {
    __shared__ float part[WAVES - 1][MB][4][64];
    if (wave > 0) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave - 1][m][i][lane] = acc[m][i];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int v = 0; v < WAVES - 1; ++v)
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[m][i] += part[v][m][i][lane];
  }
#pragma unroll
  for (int m = 0; m < MB; ++m)
    rows_f32_store<MODE>({acc[m][0], acc[m][1], acc[m][2], acc[m][3]}, block, 16 * m + r, g, bias, y, M, N, rotary);
}

// ---- the same through LDS

// A workgroup owns 16 WAVES rows of W (16 a wave), 16 MB rows of x and a slice of K. Stages of 64 k, whole lines
// of W and x, go straight from memory into LDS, DEPTH of them under way. The products of a stage start 16 / MB sums each, which
// are added in pairs; four totals take the stages in turn, so that the result is no further from 64 bits than the other kernel's
// (1.0e-7 of it for [1536, 8960], where that has 1.2e-7 to 1.5e-7).
template <int MB, int WAVES, int DEPTH, int MODE>
__global__ __launch_bounds__(64 * WAVES) void rows_f32_tiles_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                             int K, int steps_per_slice, RotaryOut rotary) {
  constexpr int ROW = RF_STEP * 4, X_BYTES = 16 * MB * ROW, SLOT = X_BYTES + 16 * WAVES * ROW, CHAINS = 16 / MB;
  constexpr int X_LOADS = (4 * MB + WAVES - 1) / WAVES, LOADS = X_LOADS + 4;       // of a wave; some of x are asked for twice
  static_assert((DEPTH + 1) * SLOT <= 160 * 1024, "LDS of a compute unit");
  __shared__ __attribute__((aligned(1024))) char lds[(DEPTH + 1) * SLOT];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), r = lane % 16, g = lane / 16;
  const int s_begin = blockIdx.y * steps_per_slice, steps = min(K / RF_STEP - s_begin, steps_per_slice);
  const int block = blockIdx.x * WAVES + wave;                 // of 16 rows of W
  // Four rows of 256 bytes a load; piece p of a row lies at place p ^ (row % 16), so that the sixteen rows a product reads at once
  // spread over all banks. Rows beyond the last are read from it and dropped.
  const float* x_lane[X_LOADS];
#pragma unroll
  for (int p = 0; p < X_LOADS; ++p) {
    const int row = 4 * ((wave * X_LOADS + p) % (4 * MB)) + lane / 16;
    x_lane[p] = x + static_cast<int64_t>(min(row, M - 1)) * K + 4 * ((lane % 16) ^ (row % 16));
  }
  const float* w_lane[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int i = 4 * p + lane / 16;
    int64_t of;
    if constexpr (MODE == PK_GATED) {
      const int half = N / 2, j = min(8 * block + i % 8, half - 1);
      of = i < 8 ? j : half + j;
    } else {
      of = min(16 * block + i, N - 1);
    }
    w_lane[p] = w + of * K + 4 * ((lane % 16) ^ i);
  }
  const uint32_t base = lds_place(lds);
  auto bring = [&](int step, int slot) {                       // (past the last step: it once more, so that the count stays)
    const int k = RF_STEP * (s_begin + min(step, steps - 1));
    const uint32_t to = base + slot * SLOT;
#pragma unroll
    for (int p = 0; p < X_LOADS; ++p) load_to_lds(x_lane[p] + k, to + (wave * X_LOADS + p) % (4 * MB) * 1024);
#pragma unroll
    for (int p = 0; p < 4; ++p) load_to_lds(w_lane[p] + k, to + X_BYTES + (wave * 4 + p) * 1024);
  };
  floatx4 total[4][MB];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int m = 0; m < MB; ++m) total[c][m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < DEPTH; ++s) bring(s, s);
  int slot = 0, s = 0;
  auto step = [&](int turn) {
    lds_arrived<(DEPTH - 1) * LOADS>();
    bring(s + DEPTH, slot == 0 ? DEPTH : slot - 1);
    const char* from = lds + slot * SLOT;
    floatx4 b[MB][4];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) b[m][j] = *reinterpret_cast<const floatx4*>(from + (16 * m + r) * ROW + 16 * ((4 * j + g) ^ r));
    floatx4 a[4], sum[CHAINS][MB];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      a[j] = *reinterpret_cast<const floatx4*>(from + X_BYTES + (16 * wave + r) * ROW + 16 * ((4 * j + g) ^ r));
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
      for (int m = 0; m < MB; ++m) sum[c][m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          floatx4& c = sum[(4 * j + e) % CHAINS][m];
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][e], b[m][j][e], c, 0, 0, 0);
        }
#pragma unroll
    for (int m = 0; m < MB; ++m) {
#pragma unroll
      for (int half = CHAINS / 2; half >= 1; half /= 2)
#pragma unroll
        for (int c = 0; c < half; ++c) sum[c][m] += sum[c + half][m];
      total[turn][m] += sum[0][m];
    }
    slot = slot == DEPTH ? 0 : slot + 1, ++s;
  };
  while (s + 4 <= steps) {
    step(0);
    step(1);
    step(2);
    step(3);
  }
  if (s < steps) step(0);
  if (s < steps) step(1);
  if (s < steps) step(2);
  lds_arrived<0>();                                                // nothing is under way when the workgroup ends
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const floatx4 acc = (total[0][m] + total[1][m]) + (total[2][m] + total[3][m]);
    rows_f32_store<MODE>({acc[0], acc[1], acc[2], acc[3]}, block, 16 * m + r, g, bias, y, M, N, rotary);
  }
}

// Slices of K: workgroups for every compute unit several times over, each at least three steps long.
void rows_plan(int row_blocks, int K, int* slices, int* steps) {
  const int all = K / RF_STEP;
  int want = 1;
  while (want < 16 && row_blocks * want < 640 && all / (want * 2) >= 3) want *= 2;
  *steps = (all + want - 1) / want;
  *slices = (all + *steps - 1) / *steps;
}

// Which products go through LDS, and how: waves of a workgroup (0: none) and slices of K. What counts is that every compute unit
// has one workgroup that asks for W and no unit two: as many waves as that takes where K stays whole, or K cut until the workgroups
// are about as many as the units (twice as many from 17 rows on, where a stage takes longer). Timed with the reader of the slices
// (us, this way / the other; every weight from memory):
//  * gated, weights of 24 million elements and more whose blocks of 16 rows make workgroups of four waves on every unit, from 12
//    rows on, from eight with K of 1,536 and more: [8, 1536] x [17920, 1536] 27.7 / 28.6, [4, 1536] 26.3 / 25.8, [32, 1536] 35 / 46; [16,
//    2048] x [16384, 2048] 32.9 / 35.0, [8, 2048] 33.0 / 31.3; [16, 1024] x [24576, 1024] 27.0 / 28.2, [8, 1024] 27.3 / 25.4. From 96 million on
//    always: [1, 3584] x [37888, 3584] 100 / 124, [8, 3584] 99 / 139, [32, 3584] 114 / 223. With fewer blocks units are idle, or three
//    waves have too little under way: [8, 4096] x [8192, 4096] 48 / 30, [8, 8192] x [4096, 8192] 87 / 33, [8, 3072] x [12288, 3072] 41 / 34.
//    Smaller weights are not: [16, 1024] x [8192, 1024] 15.0 / 12.2;
//  * plain, weights of 12 million elements and more, from eight rows on: [8, 3584] x [3584, 3584] 18.8 / 21.7, [32, 3584] 21.8 / 27.7,
//    [4, 3584] 20.9 / 20.8; up to 15 rows not where every unit would have one: some then get two, others none ([8, 4096] x [4096, 4096]
//    24.0 / 22.3, [8, 2048] x [8192, 2048] 25.4 / 23.8, [8, 11008] x [4096, 11008] 50 / 45; [8, 5120] x [5120, 5120], 240 workgroups, 28 / 34).
//    With K at least four times as long always: [1, 8960] x [1536, 8960] 18.6 / 20.3, [8, 18944] x [3584, 18944] 58 / 68, [32, 18944] 63 /
//    109. Smaller ones are level: [16, 4096] x [1024, 4096] 11.1 / 11.6, [8, 1536] x [1536, 1536] 9.0 / 8.6.
struct RowsTiles {
  int waves, slices;
};
RowsTiles rows_tiles(int M, int N, int K, bool gated) {
  const int64_t elements = static_cast<int64_t>(N) * K;
  const int blocks = gated ? (N / 2 + 7) / 8 : (N + 15) / 16, all = K / RF_STEP;
  if (gated) {
    const int waves = (blocks + 255) / 256;
    if (waves < 4 || waves > 10) return {0, 1};
    if (elements < (int64_t{96} << 20) &&
        (elements < (int64_t{24} << 20) || M < 8 || (M < 12 && (blocks <= 1024 || K < 1536))))
      return {0, 1};
    return {waves <= 5 ? waves : waves <= 7 ? 7 : 10, 1};
  }
  if (elements < (int64_t{12} << 20) || (M < 8 && K < 4 * N)) return {0, 1};
  const int groups = (blocks + 3) / 4;
  const int want = std::max(1, std::min((M <= 16 ? 256 : 512) / groups, all / 4));
  const int steps = (all + want - 1) / want;
  const int slices = (all + steps - 1) / steps;
  if (M < 16 && K < 4 * N && groups * slices > 240) return {0, 1};
  return {4, slices};
}

template <int MODE>
int launch_rows_tiles(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int row_blocks,
                      RowsTiles tiles, const RotaryOut& rotary, hipStream_t stream) {
  const dim3 grid((row_blocks + tiles.waves - 1) / tiles.waves, tiles.slices);
  const int all = K / RF_STEP, steps = (all + tiles.slices - 1) / tiles.slices;
#define TILES(WAVES, DEPTH, DEPTH2)                                                                                          \
  case WAVES:                                                                                                               \
    if (M <= 16)                                                                                                            \
      rows_f32_tiles_kernel<1, WAVES, DEPTH, MODE>                                                                          \
          <<<grid, 64 * WAVES, 0, stream>>>(x, w, bias, y, M, N, K, steps, rotary);                                         \
    else                                                                                                                    \
      rows_f32_tiles_kernel<2, WAVES, DEPTH2, MODE>                                                                         \
          <<<grid, 64 * WAVES, 0, stream>>>(x, w, bias, y, M, N, K, steps, rotary);                                         \
    break
  if constexpr (MODE == PK_PLAIN) {
    switch (tiles.waves) {
      TILES(4, 3, 2);
      default: return DISTIE_BAD_ARGUMENT;
    }
  } else {
    switch (tiles.waves) {
      TILES(4, 3, 2);
      TILES(5, 3, 3);
      TILES(7, 3, 2);
      TILES(10, 2, 2);
      default: return DISTIE_BAD_ARGUMENT;
    }
  }
#undef TILES
  return launch_status();
}

template <int MODE, int WAVES>
int launch_rows_f32(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int row_blocks, int slices,
                    int steps, const RotaryOut& rotary, hipStream_t stream) {
  const dim3 grid(row_blocks, slices);
#define ROWS(MB) rows_f32_kernel<MB, MODE, WAVES><<<grid, 64 * WAVES, 0, stream>>>(x, w, bias, y, M, N, K, steps, rotary)
  if (M <= 16) ROWS(1);
  else ROWS(2);
#undef ROWS
  return launch_status();
}

bool takes(int M, int N, int K) { return M <= 32 && N >= 1 && K >= RF_STEP && K % RF_STEP == 0; }

}  // namespace

// How many slices distie_rows_f32 writes for this weight (0: it does not take it). `whole`: not to be cut.
extern "C" int distie_rows_f32_slices(int M, int N, int K, int whole) {
  if (!takes(M, N, K)) return 0;
  int slices = 1, steps;
  if (!whole) {
    const RowsTiles tiles = rows_tiles(M, N, K, false);
    if (tiles.waves > 0) return tiles.slices;
    rows_plan((N + 15) / 16, K, &slices, &steps);
  }
  return slices;
}

// The waves of a workgroup where such a product goes through LDS, 0 where it does not.
extern "C" int distie_rows_f32_waves(int M, int N, int K, int gated) {
  return takes(M, N, K) ? rows_tiles(M, N, K, gated != 0).waves : 0;
}

// mode 0: y [M, N], or [slices, M, N] if the plan cuts K; 1 | (activation << 8): gated, [M, N / 2] (limit, slope, up_shift:
// of the clamped activation, 5); both as the products on packed copies. Up to 32 rows of x.
extern "C" int distie_rows_f32(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int mode,
                               int slices, float limit, float slope, float up_shift, hipStream_t stream) {
  if (M <= 0) return 0;
  const int act = mode >> 8;
  mode &= 0xff;
  if (!takes(M, N, K) || mode > 1 || (mode == 1 && (N % 2 != 0 || bias != nullptr || slices != 1)) || act < 0 || act > 5 ||
      (act == 5 && !(limit > 0.f)) || slices < 1)
    return DISTIE_BAD_ARGUMENT;
  RotaryOut none = {};
  none.act = act, none.limit = limit, none.slope = slope, none.up_shift = up_shift;
  const int all = K / RF_STEP, steps = (all + slices - 1) / slices;
  if ((all + steps - 1) / steps != slices) return DISTIE_BAD_ARGUMENT;
  const RowsTiles tiles = rows_tiles(M, N, K, mode == 1);
  const bool through_lds = tiles.waves > 0 && tiles.slices == slices &&
                           (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0;
  if (mode == 1) {
    const int blocks = (N / 2 + 7) / 8;
    if (through_lds) return launch_rows_tiles<PK_GATED>(x, w, nullptr, y, M, N, K, blocks, tiles, none, stream);
    if (blocks < 2048) return launch_rows_f32<PK_GATED, 4>(x, w, nullptr, y, M, N, K, blocks, 1, all, none, stream);
    return launch_rows_f32<PK_GATED, 1>(x, w, nullptr, y, M, N, K, blocks, 1, all, none, stream);
  }
  const int blocks = (N + 15) / 16;
  if (through_lds) return launch_rows_tiles<PK_PLAIN>(x, w, bias, y, M, N, K, blocks, tiles, none, stream);
  if (slices == 1 && blocks < 1024) return launch_rows_f32<PK_PLAIN, 4>(x, w, bias, y, M, N, K, blocks, 1, all, none, stream);
  return launch_rows_f32<PK_PLAIN, 1>(x, w, bias, y, M, N, K, blocks, slices, steps, none, stream);
}

// The stacked q/k/v product with bias, rotation and cache write: w [(heads + 2 kv_heads) * dim, K] as stored, table
// [M, dim / 2] (cos, sin), y [M, N] and the caches in float32.
extern "C" int distie_rows_f32_rotary(const float* x, const float* w, const float* bias, float* y, const void* table,
                                      const int32_t* slots, void* k_cache, void* v_cache, int M, int K, int heads, int kv_heads,
                                      int dim, int block_size, int write, hipStream_t stream) {
  if (M <= 0) return 0;
  const int N = (heads + 2 * kv_heads) * dim;
  if (!takes(M, N, K) || heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 != 0 || block_size < 1 || table == nullptr ||
      (write && (slots == nullptr || k_cache == nullptr || v_cache == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const RotaryOut rotary = {static_cast<const float2*>(table), slots, static_cast<bf16_t*>(k_cache),
                            static_cast<bf16_t*>(v_cache), heads, kv_heads, dim, block_size, write};
  const int all = K / RF_STEP;
  if (all >= 16) return launch_rows_f32<PK_ROTARY, 8>(x, w, bias, y, M, N, K, N / 16, 1, all, rotary, stream);
  return launch_rows_f32<PK_ROTARY, 4>(x, w, bias, y, M, N, K, N / 16, 1, all, rotary, stream);
}

