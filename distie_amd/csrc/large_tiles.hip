// Products of 9 rows and more (batches of decoding requests, prompts and portions of them) on packed weight copies: y[M, N] =
// x[M, K] W[N, K]^T for bfloat16 x and the copies of packed.h, with the activation, or rotation and cache write, in the epilogue.
//
// A workgroup of four or two waves owns a tile of rows of x and rows of W and one slice of K; a wave owns 32 TM x 32 TN of it as
// TM x TN products of 32 x 32 x 16, whose sums stay in the accumulation registers. x and W both go straight from memory into LDS:
// x in stages of 64 k (whole lines of 128 bytes: halves cost the L2 twice the requests), W, whose copy lies in lane order, in halves
// of a stage. The waits count loads, so that D stages (2, and up to 6 where tiles are small) are under way all the time; reads of
// LDS and loads stand between the matrix instructions of the 16 k before.
//
// What bounds it. [4096, 4096] x [4096, 4096] takes 110 us (1,244 TFLOP/s; the library 98): the matrix cores are 90 % busy and the
// chip's power holds the clock at 1.45 GHz, 2,270 cycles a stage, 100 us for the loop. Eight waves of 128 x 64, which read half as
// much again from LDS, needed 2,530 to 2,940 cycles at 1.58 to 1.81 GHz, 102 to 104 us whatever the cycles. That is why a wave
// owns as much as it can hold. Smaller tiles run into the L2, which gives the chip's LDS 15 to 17 TB/s: 128 x 128 need 32 KB for 512
// cycles of products (fragments of a whole stage read ahead changed nothing). With few rows it is the weight from memory: 64 rows
// of the 1.5B shape's gate+up 15.5 us (3.6 TB/s; 20.5 in packed_tiles), of the 7B shape's 53 (5.1 TB/s; 66 in passes).
// 1.5B shape, 2,048 rows, isolated and with the kernel that the library needs behind its own: gate+up with its activation 111 us
// (129), down in four slices 54 (80; the norm reads 12 us more). 7B shape, 2,048 rows: 451 (570) and 220 (359; packed_tiles
// 261). 301 rows: gate+up of the 1.5B shape 27 us, 35 in packed_tiles.

#include "common.h"
#include "lds_load.h"
#include "packed.h"
#include <algorithm>

namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

constexpr int LT_K = 64;              // k of a stage of x; W comes in halves of it
constexpr int LT_EACH = 3;            // a mode beside PK_PLAIN, PK_GATED and PK_ROTARY
constexpr int LT_EACH_MAX = 8;

// exp(-z) by 2^n 2^f, n whole: log2(e) in two parts, so that f, at most a half, keeps what a rounded product loses (with the
// contractions that the compiler would make it is off by tens of units at |z| of 30). The bounds on z keep infinities out of the
// differences and lie beyond those of the result. The same bits as expf, whose own ends of the range take four instructions more.
__device__ __forceinline__ float minus_exp(float z) {
#pragma clang fp contract(off)
  const float s = __builtin_amdgcn_fmed3f(z, -160.f, 160.f), high = -1.44269502162933349609375f * s, n = __builtin_rintf(high);
  const float low = fmaf(-1.925962991e-8f, s, fmaf(-1.44269502162933349609375f, s, -high));
  const float whole = high - n, f = whole + low;
  return __builtin_ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(n));
}

// g sigmoid(z), as g / (1 + exp(-z)) and to the same error: 0.67 units of 2^-24 in the mean and 3 at most, over |z| up to 88. The
// quotient is the unit's reciprocal and one correction, a quarter of 1 + exp(-z) because the unit flushes a reciprocal below
// 2^-126 to zero; the last instruction has the quotient of infinities and of what is no number. expf and a true division take
// longer ([2048, 1536] x [17920, 1536]: 154 us, with this quotient 113, this way 111; without the correction and with exp2(-1.4427 z)
// 104, but off by 65 units).
__device__ __forceinline__ float times_sigmoid(float g, float z) {
  const float d = fmaf(0.25f, minus_exp(z), 0.25f), n = 0.25f * g, r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, n), r, q), d, n);
}

// The workgroups of a launch: workgroup i runs on die i % 8 and every die gets a run of neighbouring tiles, the rows of x
// fastest, so that the tiles at work on a die share W and x through its L2.
struct LargePlace {
  int row_blocks;               // blocks of 16 rows of the packed copy
  int m_tiles, n_tiles, slices;
  int stages;                   // of a slice
  // LT_EACH: several weights one behind the other in one copy, each with an x of its own; what lies before the end of each
  int tile_end[LT_EACH_MAX], block_end[LT_EACH_MAX];
};

// A workgroup: WM x WAVES / WM waves of TM x TN products of 32 x 32; D stages ahead. MODE: PK_PLAIN, PK_GATED, PK_ROTARY,
// LT_EACH (plain, no bias). K a multiple of LT_K; columns of y a multiple of 16 bytes.
template <int WAVES, int WM, int TM, int TN, int D, int MODE, typename Y>
__global__ __launch_bounds__(64 * WAVES, TM * TN > 8 ? 1 : 2) void large_tiles_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias, Y* __restrict__ y, int M, int N,
    int K, LargePlace at, RotaryOut rotary) {
  constexpr int BM = 32 * WM * TM, BN = 32 * (WAVES / WM) * TN;
  constexpr int X_LOADS = BM / (8 * WAVES), W_LOADS = BN / (16 * WAVES);     // of a wave: of a stage of x, of half a stage of W
  constexpr int XA = (X_LOADS + 1) / 2, XB = X_LOADS - XA;
  constexpr int X_BYTES = BM * LT_K * 2, W_BYTES = BN * LT_K;
  constexpr int W_AT = (D + 1) * X_BYTES;
  constexpr int LDS_BYTES = W_AT + 2 * D * W_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a compute unit");
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r = lane % 32, h = lane / 32;
  const int wm = wave % WM, wn = wave / WM;
  const int tiles = at.m_tiles * at.n_tiles;
  const int place = static_cast<int>(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (place >= tiles * at.slices) return;
  const int slice = place / tiles, n_tile = place % tiles / at.m_tiles, m_tile = place % at.m_tiles;
  const int m0 = m_tile * BM;
  int b0 = n_tile * (BN / 16), block_end = at.row_blocks;
  if constexpr (MODE == LT_EACH) {
    int e = 0, tile = 0, block = 0;
    for (; n_tile >= at.tile_end[e]; ++e) tile = at.tile_end[e], block = at.block_end[e];
    b0 = block + (n_tile - tile) * (BN / 16), block_end = at.block_end[e];
    x += static_cast<int64_t>(e) * M * K;
  }
  const int s_begin = slice * at.stages;
  const int stages = min(K / LT_K - s_begin, at.stages);
  const int k_tiles = K / 32;

  const int rows = min(M - m0, BM), blocks = min(block_end - b0, BN / 16);
  const intx4 x_buffer = buffer_of(x + static_cast<int64_t>(m0) * K, static_cast<uint32_t>(rows) * K * 2u);
  const intx4 w_buffer =
      buffer_of(w + static_cast<int64_t>(b0) * k_tiles * PK_TILE, static_cast<uint32_t>(blocks) * k_tiles * 1024u);
  // A row of x's stage is eight pieces of 16 bytes; eight neighbouring lanes bring a row, piece p to place p ^ (row / 2 % 8), so
  // that the rows a product reads at once spread over all banks. Rows and blocks beyond the last are read from it and dropped.
  int x_lane[X_LOADS], w_lane[W_LOADS];
#pragma unroll
  for (int p = 0; p < X_LOADS; ++p) {
    const int row = 8 * (wave * X_LOADS + p) + lane / 8;
    x_lane[p] = min(row, rows - 1) * K * 2 + 16 * ((lane % 8) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int p = 0; p < W_LOADS; ++p) w_lane[p] = min(wave * W_LOADS + p, blocks - 1) * k_tiles * 1024 + lane * 16;
  const uint32_t base = lds_place(lds);
  auto bring_x = [&](int stage, int slot, int p) {
    buffer_to_lds(x_buffer, x_lane[p], (s_begin + min(stage, stages - 1)) * (LT_K * 2),
                  base + slot * X_BYTES + (wave * X_LOADS + p) * 1024);
  };
  auto bring_w = [&](int part, int slot, int p) {
    buffer_to_lds(w_buffer, w_lane[p], (2 * s_begin + min(part, 2 * stages - 1)) * 1024,
                  base + W_AT + slot * W_BYTES + (wave * W_LOADS + p) * 1024);
  };

  // acc[a][b][4 q + i]: row 8 (q % 2) + 4 h + i of block first_block + 2 b + q / 2, row 32 a + r of the wave's part of x
  floatx16 acc[TM][TN];
  const int first_block = b0 + wn * TN * 2;
#pragma unroll
  for (int b = 0; b < TN; ++b) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float4 start = {0.f, 0.f, 0.f, 0.f};
      if constexpr (MODE == PK_PLAIN || MODE == PK_ROTARY) {
        const int block = first_block + 2 * b + q / 2;
        const int column = MODE == PK_ROTARY ? rotary_column(block, 2 * (q % 2) + h, rotary.heads + rotary.kv_heads, rotary.dim)
                                             : 16 * block + 8 * (q % 2) + 4 * h;
        if (bias != nullptr && slice == 0 && block < at.row_blocks && column < N)
          start = *reinterpret_cast<const float4*>(bias + column);
      }
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        acc[a][b][4 * q] = start.x, acc[a][b][4 * q + 1] = start.y;
        acc[a][b][4 * q + 2] = start.z, acc[a][b][4 * q + 3] = start.w;
      }
    }
  }

  const int x_row = (wm * TM * 32 + r) * (LT_K * 2), x_turn = (r >> 1) & 7;
  bf16x8 fx[2][TM], fw[2][TN];
  const int w_at = W_AT + (wn * TN * 2 + r / 16) * 1024 + (h * 16 + r % 16) * 16;
  auto read = [&](int t, int x_slot, int w_slot, int set, int i) {
    if (i < TN)
      fw[set][i] = *reinterpret_cast<const bf16x8*>(lds + w_slot * W_BYTES + w_at + 2 * i * 1024 + t % 2 * 512);
    else
      fx[set][i - TN] = *reinterpret_cast<const bf16x8*>(lds + x_slot * X_BYTES + x_row + 16 * ((2 * t + h) ^ x_turn) +
                                                         (i - TN) * 32 * LT_K * 2);
  };
  // The products of set `set`; between them the reads of the next 16 k, and `loads` loads into LDS.
  auto multiply = [&](int set, int t, int x_slot, int w_slot, int loads, auto&& load) {
    constexpr int ALL = TM * TN, READS = TM + TN;
#pragma unroll
    for (int i = 0; i < ALL; ++i) {
      const int b = i / TM, a = i % TM;
      acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[set][b], fx[set][a], acc[a][b], 0, 0, 0);
#pragma unroll
      for (int q = i * READS / ALL; q < (i + 1) * READS / ALL; ++q) read(t, x_slot, w_slot, 1 - set, q);
#pragma unroll
      for (int q = i * loads / ALL; q < (i + 1) * loads / ALL; ++q) load(q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Past the last stage the loads bring it once more, so that their number, which the waits count, stays what it is.
#pragma unroll
  for (int p = 0; p < X_LOADS; ++p) bring_x(0, 0, p);
#pragma unroll
  for (int part = 0; part < 2 * D; ++part) {
#pragma unroll
    for (int p = 0; p < W_LOADS; ++p) bring_w(part, part, p);
#pragma unroll
    for (int p = 0; p < X_LOADS; ++p)
      if (part > 0 && part < 2 * D - 1 && (part % 2 == 1) == (p < XA)) bring_x((part + 1) / 2, (part + 1) / 2, p);
  }
  constexpr int STAGE = 2 * W_LOADS + X_LOADS;
  lds_arrived<(D - 1) * STAGE + W_LOADS>();
#pragma unroll
  for (int i = 0; i < TM + TN; ++i) read(0, 0, 0, 0, i);
  // Iteration s holds x(s) and W's parts 2 s and 2 s + 1. The loads in order: x(0), W(0); then, for every stage, W(2 s - 1), the
  // first half of x(s), W(2 s), the rest of x(s). Before the first wait W(2 s + 1) has to be there, before the second x(s + 1) and
  // W(2 s + 2); D stages have been asked for. A wait also says that all waves have read what the loads behind it write over.
  int slot = 0, w_slot = 0;
  for (int s = 0; s < stages; ++s) {
    const int next = slot == D ? 0 : slot + 1, free = slot == 0 ? D : slot - 1, w_next = w_slot == 2 * D - 2 ? 0 : w_slot + 2;
    multiply(0, 1, slot, w_slot, XA, [&](int q) { bring_x(s + D, free, q); });
    lds_arrived<(D - 1) * STAGE + XA>();
    multiply(1, 2, slot, w_slot + 1, W_LOADS, [&](int q) { bring_w(2 * (s + D), w_slot, q); });
    multiply(0, 3, slot, w_slot + 1, XB, [&](int q) { bring_x(s + D, free, XA + q); });
    lds_arrived<(D - 1) * STAGE>();
    multiply(1, 0, next, w_next, W_LOADS, [&](int q) { bring_w(2 * (s + D) + 1, w_slot + 1, q); });
    slot = next, w_slot = w_next;
  }
  lds_arrived<0>();

  // The results of 32 rows of x and up to 128 bytes of columns at a time go through LDS, so that rows leave in whole lines.
  constexpr int EACH = MODE == PK_GATED ? 16 : 32;                                  // columns of y that 32 rows of W give
  constexpr int GROUP = 128 / (EACH * static_cast<int>(sizeof(Y)));                 // so many blocks of 32 at a time
  constexpr int STRIDE = 128 + 16, PIECE = 16 / static_cast<int>(sizeof(Y));        // bytes of a row there; values of a store
  char* own = lds + wave * (32 * STRIDE);
  const int columns = MODE == PK_GATED ? N / 2 : N, column_end = MODE == LT_EACH ? 16 * block_end : columns;
  const int column0 = first_block * (MODE == PK_GATED ? 8 : 16);
  Y* out = y + static_cast<int64_t>(slice) * M * N;
  const int half = rotary.dim / 2, per_head = rotary.dim / 16, turned = rotary.heads + rotary.kv_heads;      // (PK_ROTARY)
  // first and second: four values each of the two halves of a block, of token m; turns the pairs of q and k, and puts the values
  // into their cache, where neighbouring tokens lie side by side
  auto turn = [&](float* first, float* second, int m, int block) {
    const int head = block / per_head, sub = block % per_head;
    if (head < turned) {
      const float4* angles =
          reinterpret_cast<const float4*>(rotary.table + static_cast<int64_t>(min(m, M - 1)) * half + 8 * sub + 4 * h);
      const float4 low = angles[0], high = angles[1];
      const float c[4] = {low.x, low.z, high.x, high.z}, s[4] = {low.y, low.w, high.y, high.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float one = first[i], two = second[i];
        first[i] = one * c[i] - two * s[i];
        second[i] = two * c[i] + one * s[i];
      }
    } else if (rotary.write && m < M && block < at.row_blocks) {
      const int slot = rotary.slots[m];
      const int64_t page = slot / rotary.block_size, row = 16 * sub + 4 * h;
      Y* value = reinterpret_cast<Y*>(rotary.v_cache) +
                 ((page * rotary.kv_heads + head - turned) * rotary.dim + row) * rotary.block_size + slot % rotary.block_size;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        value[static_cast<int64_t>(i) * rotary.block_size] = from_float<Y>(first[i]);
        value[static_cast<int64_t>(8 + i) * rotary.block_size] = from_float<Y>(second[i]);
      }
    }
  };
  auto finish = [&](auto&& gated) {
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int row0 = m0 + (wm * TM + a) * 32;
#pragma unroll
      for (int g = 0; g < TN; g += GROUP) {
        const int count = TN - g < GROUP ? TN - g : GROUP;
#pragma unroll
        for (int b = g; b < g + count; ++b) {
          char* to = own + r * STRIDE + ((b - g) * EACH + 4 * h) * sizeof(Y);
#pragma unroll
          for (int q = 0; q < 4; q += MODE == PK_GATED || MODE == PK_ROTARY ? 2 : 1) {
            float v[4], v2[4];
            if constexpr (MODE == PK_GATED) {
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] = gated(acc[a][b][4 * q + i], acc[a][b][4 * q + 4 + i]);
              *reinterpret_cast<uint2*>(to + q / 2 * 8 * sizeof(Y)) = pack_bf16x4(v);
            } else if constexpr (MODE == PK_ROTARY) {
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] = acc[a][b][4 * q + i], v2[i] = acc[a][b][4 * q + 4 + i];
              turn(v, v2, row0 + r, first_block + 2 * b + q / 2);
              *reinterpret_cast<uint2*>(to + q * 8 * sizeof(Y)) = pack_bf16x4(v);
              *reinterpret_cast<uint2*>(to + (q + 1) * 8 * sizeof(Y)) = pack_bf16x4(v2);
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] = acc[a][b][4 * q + i];
              if constexpr (sizeof(Y) == 2) *reinterpret_cast<uint2*>(to + q * 8 * sizeof(Y)) = pack_bf16x4(v);
              else *reinterpret_cast<float4*>(to + q * 8 * sizeof(Y)) = float4{v[0], v[1], v[2], v[3]};
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const int pieces = count * EACH / PIECE;           // of a row
#pragma unroll
        for (int i = 0; i < 32 * pieces / 64; ++i) {
          const int e = 64 * i + lane, row = e / pieces, piece = e % pieces;
          const uint4 v = *reinterpret_cast<const uint4*>(own + row * STRIDE + 16 * piece);
          if constexpr (MODE == PK_ROTARY) {
            // a piece is half a block: eight neighbouring columns of a head
            const int block = first_block + 2 * g + piece / 2;
            if (row0 + row < M && block < at.row_blocks) {
              const int column = rotary_column(block, 2 * (piece % 2), turned, rotary.dim);
              *reinterpret_cast<uint4*>(out + static_cast<int64_t>(row0 + row) * N + column) = v;
              const int head = block / per_head;
              if (rotary.write && head >= rotary.heads && head < turned) {
                const int slot = rotary.slots[row0 + row];
                const int64_t page = slot / rotary.block_size;
                Y* key = reinterpret_cast<Y*>(rotary.k_cache) +
                         ((page * rotary.kv_heads + head - rotary.heads) * rotary.block_size + slot % rotary.block_size) * rotary.dim;
                *reinterpret_cast<uint4*>(key + column - head * rotary.dim) = v;
              }
            }
          } else {
            const int column = column0 + g * EACH + piece * PIECE;
            if (row0 + row < M && column < column_end)
              *reinterpret_cast<uint4*>(out + static_cast<int64_t>(row0 + row) * columns + column) = v;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    }
  };
  if (MODE == PK_GATED && rotary.act == 0) {
    finish([&](float gate, float up) { return times_sigmoid(gate, gate) * up; });
  } else if (MODE == PK_GATED && rotary.act == 5) {
    finish([&](float gate, float up) {
      const float g = fminf(gate, rotary.limit), u = fminf(fmaxf(up, -rotary.limit), rotary.limit);
      return times_sigmoid(g, rotary.slope * g) * (u + rotary.up_shift);
    });
  } else if (MODE == PK_GATED && rotary.act == 3) {
    // 0.5 z (1 + tanh u) = z sigmoid(2 u): nothing cancels, and tanhf took three times as long as expf and the quotient
    finish([&](float gate, float up) {
      return times_sigmoid(gate, 1.5957691216057308f * (gate + 0.044715f * gate * gate * gate)) * up;
    });
  } else {
    // (a choice among all activations for every value took 40 % more than this one between two)
    finish([&](float gate, float up) {
      const float p = fmaxf(gate, 0.f);
      return (rotary.act == 1 ? p * p : p) * up;
    });
  }
}

// The tiles there are, and what a workgroup of one of the first takes: for every stage few_us with hardly any compute unit at
// work, more_us on top of it with all of them (the L2; and power: the clock falls from 2.4 to 1.45 GHz) and pair_us where two
// share them, and turn_us to begin and end. The others are for few rows (`plan_few`).
struct LargeShape {
  int waves, wm, tm, tn;
  float few_us, more_us, pair_us, turn_us;

  constexpr int rows() const { return 32 * wm * tm; }
  constexpr int blocks() const { return 2 * (waves / wm) * tn; }
};
constexpr LargeShape LARGE_SHAPES[] = {
    {4, 2, 4, 4, 0.893f, 0.515f, 0.f, 6.7f},  {4, 2, 4, 3, 0.684f, 0.451f, 0.f, 5.3f},
    {4, 2, 3, 4, 0.692f, 0.446f, 0.f, 5.7f},  {4, 2, 3, 3, 0.558f, 0.371f, 0.f, 4.3f},
    {4, 2, 2, 4, 0.528f, 0.373f, 0.f, 3.4f},  {4, 2, 3, 2, 0.386f, 0.317f, 0.f, 2.7f},
    {4, 2, 2, 3, 0.407f, 0.327f, 0.f, 2.55f}, {4, 2, 2, 2, 0.280f, 0.336f, 0.497f, 1.8f},
    {4, 1, 1, 1}, {4, 1, 1, 2}, {4, 1, 2, 1}, {4, 2, 1, 1}, {2, 1, 1, 1}, {2, 1, 2, 1}};
constexpr int LARGE_COUNTED = 8, FEW_32_128 = 8, FEW_32_256 = 9, FEW_64_128 = 10, FEW_64_64 = 11, FEW_32_64 = 12, FEW_64_64_CUT = 13;
constexpr int LARGE_ROTARY_FROM = 1, LARGE_ROTARY_TO = LARGE_COUNTED;          // (the sums and angles of the first do not fit the registers)
constexpr int LARGE_SHAPE_COUNT = static_cast<int>(sizeof(LARGE_SHAPES) / sizeof(LARGE_SHAPES[0]));
constexpr float LARGE_GATED_TURN = 0.81f, LARGE_ROTARY_TURN = 3.4f;     // (half the stores; angles and the caches' stores)

struct LargePlan {
  int shape, slices;
  float us;
};

// How a product is cut, as plan_tiles: whole rounds of workgroups on the compute units, the last of them with as many as are
// left, no faster than memory brings W, and what the reader of the result moves. The numbers are a least-squares fit to 16,000
// timings (25 weights of 0.9 to 136 million elements, 65 to 2,048 rows, in a captured graph; it is off by 6 %), but for two that
// it could not tell: what a second workgroup costs a unit, and the rate of W from memory where rows are few, 5.2 TB/s. What the
// count chooses takes 1.6 % more than the best of them on average, a tenth and more in 24 cases of 655.
LargePlan plan_large(int M, int N, int K, int row_blocks, int mode, bool may_cut, float cut_us) {
  LargePlan best = {-1, 0, 0.f};
  const int all = K / LT_K;
  const float memory_us = static_cast<float>(row_blocks) * K * 32.f / 5.2e6f, values = static_cast<float>(M) * N;
  for (int i = 0; i < LARGE_COUNTED; ++i) {
    const LargeShape& s = LARGE_SHAPES[i];
    if (mode == PK_ROTARY && (i < LARGE_ROTARY_FROM || i >= LARGE_ROTARY_TO)) continue;
    const int64_t tiles = static_cast<int64_t>((M + s.rows() - 1) / s.rows()) * ((row_blocks + s.blocks() - 1) / s.blocks());
    const float turn = s.turn_us * (mode == PK_GATED ? LARGE_GATED_TURN : mode == PK_ROTARY ? LARGE_ROTARY_TURN : 1.f);
    for (int cut = 1; cut <= 8; ++cut) {
      if (cut > 1 && (!may_cut || all / cut < 6)) break;
      const int stages = (all + cut - 1) / cut;
      if ((all + stages - 1) / stages != cut) continue;
      const int64_t units = s.pair_us > 0.f ? 512 : 256, work = tiles * cut, full = work / units, rest = work % units;
      const float busy = rest / 256.f;
      float us = full * (stages * (s.few_us + s.more_us + s.pair_us) + turn);
      // (a unit with two takes its time however few such units there are, by how loaded the chip is: half of pair_us and up)
      const float pair = busy > 1.f ? s.pair_us * (0.45f + 0.5f * (busy - 1.f)) : 0.f;
      if (rest > 0) us += stages * (s.few_us + s.more_us * std::min(busy, 1.f) + pair) + turn;
      us = 2.2f + std::max(us, memory_us);
      if (cut > 1) us += 4.f * cut * values / 8.0e6f;
      if (mode == PK_PLAIN && may_cut) {
        if (cut_us == 0.f) us += std::max(3.7f, 3.8f + (4.f * cut + 10.f) * values / 8.6e6f);      // the norm that adds the slices
        else if (cut > 1) us += cut_us + (4.f * cut + 2.f) * values / 8.6e6f;
      }
      if (best.shape < 0 || us < best.us) best = {i, cut, us};
    }
  }
  return best;
}

// Few rows: the weight comes from memory once, and what counts is that every compute unit has one workgroup that asks for it and
// no unit two, which would take twice as long: the smallest tile whose workgroups are no more than the units; K cut until they
// are about as many. (us: gate+up of the 1.5B shape, 16 rows: 140 workgroups of 32 x 128 12.8, 280 of 32 x 64 15.5; [16384, 2048],
// 256 of 32 x 64 14.5, 128 of 32 x 128 18.3; [37888, 3584], 32 rows, 148 of 32 x 256 53, 296 of 32 x 128 64; 64 rows, 198 of 128 x 192
// 51.6, 592 of 64 x 64 62. [4096, 11008] in four, 64 rows: 256 of 64 x 64 25.) Beyond that many workgroups small tiles do best.
constexpr int FEW_ROWS = 64;

LargePlan plan_few(int M, int N, int K, int row_blocks, int mode, bool may_cut, float cut_us) {
  const int all = K / LT_K;
  const auto workgroups = [&](int shape) { return (row_blocks + LARGE_SHAPES[shape].blocks() - 1) / LARGE_SHAPES[shape].blocks(); };
  if (mode == PK_PLAIN && may_cut && cut_us == 0.f) {
    int shape = M <= 32 ? FEW_32_64 : FEW_64_64_CUT;
    const auto cut_for = [&](int i) { return std::max(1, std::min(256 / workgroups(i), all / 4)); };
    if (shape == FEW_64_64_CUT && all > 64 * cut_for(shape)) shape = FEW_64_128;       // long walks: wider tiles, twice as many cuts
    const int stages = (all + cut_for(shape) - 1) / cut_for(shape);
    return {shape, (all + stages - 1) / stages, 0.f};
  }
  if (M <= 32) {
    for (int shape : {FEW_32_64, FEW_32_128, FEW_32_256})
      if (workgroups(shape) <= 256) return {shape, 1, 0.f};
    return {FEW_32_64, 1, 0.f};
  }
  for (int shape : {FEW_64_64, FEW_64_128, 6, 4})             // (128 x 192 and 128 x 256)
    if (workgroups(shape) <= 256) return {shape, 1, 0.f};
  return {FEW_64_128, 1, 0.f};
}

template <int MODE, typename Y>
int launch_large(const bf16_t* x, const bf16_t* w, const float* bias, Y* y, int M, int N, int K, int row_blocks, int shape,
                 int slices, const RotaryOut& rotary, hipStream_t stream, int count = 0, const int32_t* ends = nullptr) {
  const int bm = LARGE_SHAPES[shape].rows(), blocks = LARGE_SHAPES[shape].blocks();
  const int all = K / LT_K;
  LargePlace at = {row_blocks, (M + bm - 1) / bm, (row_blocks + blocks - 1) / blocks, slices, (all + slices - 1) / slices};
  if (MODE == LT_EACH) {
    at.n_tiles = 0;
    for (int e = 0, begin = 0; e < count; begin = ends[e++]) {
      at.n_tiles += (ends[e] - begin + blocks - 1) / blocks;
      at.tile_end[e] = at.n_tiles, at.block_end[e] = ends[e];
    }
  }
  if ((all + at.stages - 1) / at.stages != slices) return DISTIE_BAD_ARGUMENT;
  const int64_t work = static_cast<int64_t>(at.m_tiles) * at.n_tiles * slices;
  if (work > (1 << 30)) return DISTIE_BAD_ARGUMENT;
  const unsigned grid = static_cast<unsigned>((work + 7) / 8 * 8);
#define LARGE(I, WAVES, WM, TM, TN, D)                                                                                    \
  case I:                                                                                                                 \
    if constexpr (MODE != PK_ROTARY || (I >= LARGE_ROTARY_FROM && I < LARGE_ROTARY_TO)) {                                 \
      static_assert(LARGE_SHAPES[I].waves == WAVES && LARGE_SHAPES[I].rows() == 32 * WM * TM &&                           \
                        LARGE_SHAPES[I].blocks() == 2 * (WAVES / WM) * TN, "the table's tile");                           \
      large_tiles_kernel<WAVES, WM, TM, TN, D, MODE, Y><<<grid, 64 * WAVES, 0, stream>>>(x, w, bias, y, M, N, K, at, rotary); \
      break;                                                                                                              \
    }                                                                                                                     \
    return DISTIE_BAD_ARGUMENT
  switch (shape) {
    LARGE(0, 4, 2, 4, 4, 2);
    LARGE(1, 4, 2, 4, 3, 2);
    LARGE(2, 4, 2, 3, 4, 2);
    LARGE(3, 4, 2, 3, 3, 2);
    LARGE(4, 4, 2, 2, 4, 2);
    LARGE(5, 4, 2, 3, 2, 2);
    LARGE(6, 4, 2, 2, 3, 2);
    LARGE(7, 4, 2, 2, 2, 2);
    LARGE(8, 4, 1, 1, 1, 3);
    LARGE(9, 4, 1, 1, 2, 3);
    LARGE(10, 4, 1, 2, 1, 3);
    LARGE(11, 4, 2, 1, 1, 3);
    LARGE(12, 2, 1, 1, 1, 6);
    LARGE(13, 2, 1, 2, 1, 3);
    default: return DISTIE_BAD_ARGUMENT;
  }
#undef LARGE
  return launch_status();
}

bool aligned(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

// How the kernels of this file cut a product, 0 if they do not take it, as distie_packed_tiles_plan. mode: 0 plain, 1 gated, 2
// with rotation and cache write; *us: what the count comes to (few rows: 0, not counted).
extern "C" int distie_large_tiles_plan(int M, int N, int K, int mode, int may_cut, float cut_us, int* shape, int* slices,
                                       float* us) {
  if (M < 1 || N < 16 || K < 4 * LT_K || K % LT_K != 0 || mode < 0 || mode > 2 || N % (mode == PK_GATED ? 16 : 8) != 0 ||
      (mode == PK_ROTARY && N % 16 != 0) || K > (1 << 20))
    return 0;
  const bool cut = may_cut != 0 && mode == PK_PLAIN;
  const LargePlan plan = M <= FEW_ROWS && mode != PK_ROTARY ? plan_few(M, N, K, (N + 15) / 16, mode, cut, cut_us)
                                                            : plan_large(M, N, K, (N + 15) / 16, mode, cut, cut_us);
  *shape = plan.shape, *slices = plan.slices, *us = plan.us;
  return 1;
}

// How many tiles of that shape lie one below the other for M rows, and side by side for N columns.
extern "C" int distie_large_tiles_grid(int M, int N, int shape, int* row_tiles, int* column_tiles) {
  if (M < 1 || N < 1 || shape < 0 || shape >= LARGE_SHAPE_COUNT) return DISTIE_BAD_ARGUMENT;
  const LargeShape& s = LARGE_SHAPES[shape];
  *row_tiles = (M + s.rows() - 1) / s.rows(), *column_tiles = ((N + 15) / 16 + s.blocks() - 1) / s.blocks();
  return 0;
}

// y: [M, N] of y_dtype (gated: [M, N / 2] in bfloat16), or with slices > 1 float32 [slices, M, N], to be added in order by
// whoever reads it, the bias in the first. All pointers at multiples of 16 bytes.
extern "C" int distie_large_tiles_bf16(const void* x, const void* w_packed, const float* bias, void* y, int y_dtype, int M,
                                       int N, int K, int gated, int shape, int slices, float limit, float slope, float up_shift,
                                       hipStream_t stream) {
  if (M <= 0) return 0;
  const int act = gated >> 8 == 2 ? 0 : gated >> 8;           // the activation on the gate, above the low eight bits (2: silu, too)
  gated &= 0xff;
  if (N < 16 || K < 4 * LT_K || K % LT_K != 0 || K > (1 << 20) || shape < 0 || shape >= LARGE_SHAPE_COUNT || slices < 1 ||
      gated > 1 || N % (gated ? 16 : 8) != 0 || (gated && (slices != 1 || y_dtype != DISTIE_BF16 || bias != nullptr)) ||
      act < 0 || act > 5 || (act == 5 && !(limit > 0.f)) || (slices > 1 && y_dtype != DISTIE_F32) || !aligned(x) ||
      !aligned(w_packed) || !aligned(bias) || !aligned(y))
    return DISTIE_BAD_ARGUMENT;
  RotaryOut out = {};
  out.act = act, out.limit = limit, out.slope = slope, out.up_shift = up_shift;
  const bf16_t* xb = static_cast<const bf16_t*>(x);
  const bf16_t* wb = static_cast<const bf16_t*>(w_packed);
  const int blocks = (N + 15) / 16;
  if (gated) return launch_large<PK_GATED, bf16_t>(xb, wb, nullptr, static_cast<bf16_t*>(y), M, N, K, blocks, shape, 1, out, stream);
  DISTIE_DISPATCH(y_dtype, Y, return (launch_large<PK_PLAIN, Y>(xb, wb, bias, static_cast<Y*>(y), M, N, K, blocks, shape, slices,
                                                                out, stream)));
  return DISTIE_BAD_ARGUMENT;
}

// The stacked q/k/v product with rotation and cache write in its epilogue, as distie_gemm_packed_rotary_bf16.
extern "C" int distie_large_tiles_rotary_bf16(const void* x, const void* w_packed, const float* bias, void* y, const void* table,
                                              const int32_t* slots, void* k_cache, void* v_cache, int M, int K, int heads,
                                              int kv_heads, int dim, int block_size, int write, int shape, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K < 4 * LT_K || K % LT_K != 0 || K > (1 << 20) || heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 != 0 || block_size < 1 ||
      shape < LARGE_ROTARY_FROM || shape >= LARGE_ROTARY_TO || table == nullptr ||
      (write && (slots == nullptr || k_cache == nullptr || v_cache == nullptr)) || !aligned(x) || !aligned(w_packed) ||
      !aligned(bias) || !aligned(y) || !aligned(table) || !aligned(k_cache))
    return DISTIE_BAD_ARGUMENT;
  const int N = (heads + 2 * kv_heads) * dim;
  const RotaryOut rotary = {static_cast<const float2*>(table), slots, static_cast<bf16_t*>(k_cache),
                            static_cast<bf16_t*>(v_cache), heads, kv_heads, dim, block_size, write};
  return launch_large<PK_ROTARY, bf16_t>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w_packed), bias,
                                         static_cast<bf16_t*>(y), M, N, K, N / 16, shape, 1, rotary, stream);
}

// xs [count, M, K], each with its own rows of the copy, which end at block ends[e] (the last at `blocks`): y [M, 16 blocks] in
// bfloat16, weight e in the columns that its blocks have. shape: as distie_large_tiles_plan gives it for 16 blocks columns.
extern "C" int distie_large_tiles_each_bf16(const void* xs, const void* w_packed, void* y, int M, int K, int count,
                                            const int32_t* ends, int shape, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K < 4 * LT_K || K % LT_K != 0 || K > (1 << 20) || count < 1 || count > LT_EACH_MAX || ends == nullptr || shape < 0 ||
      shape >= LARGE_SHAPE_COUNT || !aligned(xs) || !aligned(w_packed) || !aligned(y))
    return DISTIE_BAD_ARGUMENT;
  for (int e = 0; e < count; ++e)
    if (ends[e] <= (e > 0 ? ends[e - 1] : 0) || ends[e] > (1 << 24)) return DISTIE_BAD_ARGUMENT;
  return launch_large<LT_EACH, bf16_t>(static_cast<const bf16_t*>(xs), static_cast<const bf16_t*>(w_packed), nullptr,
                                       static_cast<bf16_t*>(y), M, 16 * ends[count - 1], K, ends[count - 1], shape, 1, RotaryOut{},
                                       stream, count, ends);
}
