// What the kernels on packed weight copies share: vector types of the matrix cores' operands, the tile of
// a packed copy, and the description of the q/k/v epilogue.
#pragma once

#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define PK_TILE 512         // elements of a tile: 16 rows x 32 k, in lane order
#define PK_PLAIN 0
#define PK_GATED 1
#define PK_ROTARY 2

struct RotaryOut {
  const float2* table;        // [M, D / 2] cosine and sine of each token's angles
  const int32_t* slots;       // [M] place of each token in the cache
  bf16_t* k_cache;            // [pages, kv_heads, block_size, D] (float32 behind these pointers where the result is)
  bf16_t* v_cache;            // [pages, kv_heads, D, block_size]
  int heads, kv_heads, dim, block_size, write;
  int act;                    // gated products only: the activation on the gate (see gate_activation)
  float limit, slope, up_shift;      // of the clamped one (see gated_value)
};

// The activation on the gate of a gated product: 0 silu; else 1 + the kind as `distie_activation` numbers them
// (1: the square of max(z, 0), 3: the tanh form of gelu, 4: max(z, 0)). The C interface takes it in the bits above
// the low eight of its `gated` / `mode` argument.
static __device__ __forceinline__ float gate_activation(float z, int act) {
  if (act == 0 || act == 2) return z / (1.f + expf(-z));
  if (act == 3) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  const float p = fmaxf(z, 0.f);
  return act == 1 ? p * p : p;
}

// gate and up of one hidden value put together. act 5: g = min(gate, limit), u = clamp(up, -limit, limit),
// g * sigmoid(slope * g) * (u + up_shift); else the activation of the gate times up.
static __device__ __forceinline__ float gated_value(float gate, float up, int act, float limit, float slope, float up_shift) {
  if (act != 5) return gate_activation(gate, act) * up;
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return g / (1.f + expf(-slope * g)) * (u + up_shift);
}

static __device__ __forceinline__ uint2 pack_bf16x4(const float v[4]) {
  uint32_t h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) h[i] = __builtin_bit_cast(uint16_t, static_cast<bf16_t>(v[i]));
  return uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
}

// four neighbouring values of a row, from column n0 on, of which those below `columns` exist
template <typename Y>
static __device__ __forceinline__ void store_four(Y* row, int n0, int columns, const float v[4]) {
  if (n0 + 4 <= columns && columns % 4 == 0) {
    if constexpr (sizeof(Y) == 2) *reinterpret_cast<uint2*>(row + n0) = pack_bf16x4(v);
    else *reinterpret_cast<float4*>(row + n0) = float4{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n0 + i < columns) row[n0 + i] = from_float<Y>(v[i]);
  }
}

// The first of the four columns, in the weight's own order, that lane group g holds of block `block` of a ROTARY copy:
// block (head, sub) of a q or k head holds the head's rows 8 sub .. + 7 and dim / 2 + 8 sub .. + 7, of a v head 16 in order.
static __device__ __forceinline__ int rotary_column(int block, int g, int turned_heads, int dim) {
  const int per_head = dim / 16, head = block / per_head, sub = block % per_head;
  return head * dim + (head < turned_heads ? (g / 2) * (dim / 2) + 8 * sub + 4 * (g % 2) : 16 * sub + 4 * g);
}

// The end of a q/k/v product on a ROTARY copy: sums[i] is row 4 g + i of the block for token m. Adds the bias, turns the
// pairs (partners are lanes 32 apart: every lane of the wave has to come here), writes y and the paged cache where
// `inside` says that the token exists.
template <typename Y>
static __device__ __forceinline__ void store_rotary(const float sums[4], int64_t m, bool inside, int g, int block,
                                                    const float* bias, Y* y, int N, const RotaryOut& rotary) {
  const int dim = rotary.dim, half = dim / 2, per_head = dim / 16;
  const int head = block / per_head, sub = block % per_head;          // among q, k, v heads in this order
  const bool turns = head < rotary.heads + rotary.kv_heads;
  const int column = rotary_column(block, g, rotary.heads + rotary.kv_heads, dim), d0 = column - head * dim;
  float own[4], other[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) own[i] = sums[i] + (bias != nullptr ? bias[column + i] : 0.f);
#pragma unroll
  for (int i = 0; i < 4; ++i) other[i] = __shfl_xor(own[i], 32, 64);
  if (!inside) return;
  float v[4];
  if (turns) {
    const float2* angles = rotary.table + m * half + 8 * sub + 4 * (g % 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 cs = angles[i];
      // first half: x1 cos - x2 sin; second half: x2 cos + x1 sin
      v[i] = g < 2 ? own[i] * cs.x - other[i] * cs.y : own[i] * cs.x + other[i] * cs.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = own[i];
  }
  store_four(y + m * N, column, N, v);
  if (!rotary.write || head < rotary.heads) return;
  const int slot = rotary.slots[m];                    // (divided in 32 bits: in 64 it is some hundred instructions a block)
  const int64_t page = slot / rotary.block_size;
  const int offset = slot % rotary.block_size;
  if (turns) {
    const int kv_head = head - rotary.heads;
    Y* at = reinterpret_cast<Y*>(rotary.k_cache) + ((page * rotary.kv_heads + kv_head) * rotary.block_size + offset) * dim;
    store_four(at, d0, dim, v);
  } else {
    const int kv_head = head - rotary.heads - rotary.kv_heads;
    Y* at = reinterpret_cast<Y*>(rotary.v_cache) + ((page * rotary.kv_heads + kv_head) * dim + d0) * rotary.block_size + offset;
#pragma unroll
    for (int i = 0; i < 4; ++i) at[static_cast<int64_t>(i) * rotary.block_size] = from_float<Y>(v[i]);
  }
}
