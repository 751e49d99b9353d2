// Shared helpers of the HIP kernels (gfx950, 64-wide wavefronts).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;

// dtype codes of the C interface
#define DISTIE_F32 0
#define DISTIE_BF16 1

// status codes of the C interface: 0 = launched; >0 = hipError_t; <0 = refused (bad argument)
#define DISTIE_BAD_ARGUMENT (-1)

#define DISTIE_WAVE 64

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(bf16_t x) { return static_cast<float>(x); }

template <typename T>
__device__ __forceinline__ T from_float(float x);
template <>
__device__ __forceinline__ float from_float<float>(float x) { return x; }
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float x) { return static_cast<bf16_t>(x); }  // round to nearest even

// The loads in front of it are asked for before anything behind it (left to itself the compiler puts each in front of its use).
__device__ __forceinline__ void loads_first() { __builtin_amdgcn_sched_barrier(0); }

// The values of lanes i and i ^ O, in one order or the other: whoever adds them or takes the larger has the same in both lanes. Within
// rows of 16 lanes by DPP (8: rotated by half a row; 4: each half of a row mirrored, then each quad; 2 and 1: a quad's lanes permuted),
// beyond by the swaps of 16 and 32 lanes: a step of a sum is a move and an add in the vector ALU, where `__shfl_xor` sends the
// value through the LDS unit and waits for it. All 64 lanes take part. The sums are the same bits; steps, us, so / now: one
// request of 500 keys 1,090 / 1,076, 64 requests of 2,048 keys 2,377 / 2,360, Dufelix with 16 requests 1,442 / 1,424.
struct LanePair {
  float a, b;
};
template <int O>
__device__ __forceinline__ LanePair lanes_apart(float v) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "a power of two below 64");
  const int bits = __builtin_bit_cast(int, v);
  if constexpr (O >= 16) {
    const auto both = [&] {
      if constexpr (O == 32) return __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
      else return __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    }();
    const uint32_t low = both[0], high = both[1];
    return {__builtin_bit_cast(float, low), __builtin_bit_cast(float, high)};
  } else {
    constexpr int ROTATE_8 = 0x128, MIRROR_HALVES = 0x141, MIRROR_QUADS = 0x1B, SWAP_PAIRS = 0x4E, SWAP = 0xB1;
    constexpr int FIRST = O == 8 ? ROTATE_8 : O == 4 ? MIRROR_HALVES : O == 2 ? SWAP_PAIRS : SWAP;
    int other = __builtin_amdgcn_update_dpp(0, bits, FIRST, 0xf, 0xf, true);
    if constexpr (O == 4) other = __builtin_amdgcn_update_dpp(0, other, MIRROR_QUADS, 0xf, 0xf, true);
    return {v, __builtin_bit_cast(float, other)};
  }
}
template <int O>
__device__ __forceinline__ float lanes_sum(float v) {
  const LanePair p = lanes_apart<O>(v);
  return p.a + p.b;
}
template <int O>
__device__ __forceinline__ float lanes_max(float v) {
  const LanePair p = lanes_apart<O>(v);
  return fmaxf(p.a, p.b);
}

__device__ __forceinline__ float wave_sum(float v) {
  return lanes_sum<1>(lanes_sum<2>(lanes_sum<4>(lanes_sum<8>(lanes_sum<16>(lanes_sum<32>(v))))));
}

__device__ __forceinline__ float wave_max(float v) {
  return lanes_max<1>(lanes_max<2>(lanes_max<4>(lanes_max<8>(lanes_max<16>(lanes_max<32>(v))))));
}

// Sum over a block of up to 1024 threads; `scratch` holds one float per wave (16).
// The order of the additions depends only on the block size, never on the data's place in a batch.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int waves = (blockDim.x + DISTIE_WAVE - 1) / DISTIE_WAVE;
  v = wave_sum(v);
  const int wave = threadIdx.x / DISTIE_WAVE;
  const int lane = threadIdx.x % DISTIE_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  // a few waves' places, or all sixteen, are read together, and those that no wave wrote are dropped (a loop over the waves waited for
  // each; sixteen for every block: norms of groups of 128, 2,048 rows of 2,048, 13.9 -> 14.7 us)
  float part[16];
  float total;
  if (waves <= 4) {
#pragma unroll
    for (int w = 0; w < 4; ++w) part[w] = scratch[w];
    total = part[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) total = w < waves ? total + part[w] : total;
  } else {
#pragma unroll
    for (int w = 0; w < 16; ++w) part[w] = scratch[w];
    total = part[0];
#pragma unroll
    for (int w = 1; w < 16; ++w) total = w < waves ? total + part[w] : total;
  }
  return total;
}

// Sum of `slices` values that lie `stride` elements apart, added in order. The loads of four slices are
// issued together (the last group re-reads the last slice where it has fewer than four and does not add
// it), so the sum costs a few memory round trips instead of one per slice.
template <typename T>
__device__ __forceinline__ float sum_strided(const T* p, int slices, int64_t stride) {
  float sum = 0.f;
  for (int s = 0; s < slices; s += 4) {
    const int last = slices - 1;
    const float a = to_float(p[s * stride]);
    const float b = to_float(p[min(s + 1, last) * stride]);
    const float c = to_float(p[min(s + 2, last) * stride]);
    const float d = to_float(p[min(s + 3, last) * stride]);
    loads_first();                              // (selects below: where a sum stands under a condition, its load is put there too)
    sum += a;
    sum = s + 1 <= last ? sum + b : sum;
    sum = s + 2 <= last ? sum + c : sum;
    sum = s + 3 <= last ? sum + d : sum;
  }
  return sum;
}

static inline int launch_status() { return static_cast<int>(hipGetLastError()); }

// Calls `body` with a value of the element type that `code` names.
#define DISTIE_DISPATCH(code, T, ...)                 \
  do {                                                \
    if ((code) == DISTIE_F32) {                       \
      using T = float;                                \
      __VA_ARGS__;                                    \
    } else if ((code) == DISTIE_BF16) {               \
      using T = bf16_t;                               \
      __VA_ARGS__;                                    \
    } else {                                          \
      return DISTIE_BAD_ARGUMENT;                     \
    }                                                 \
  } while (0)
