// Loads from memory straight into LDS, which the kernels that keep several stages of them under way share. Instructions of their own
// because the compiler, which knows of such loads, waits for all of them before any read of LDS: the waits are the caller's, which
// counts them (`lds_arrived`). Nothing may be under way when a workgroup ends.
#pragma once

#include "common.h"

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int intx4;

// Where in LDS `p` lies, which is the same in all lanes.
static __device__ __forceinline__ uint32_t lds_place(const void* p) {
  return __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)p)));
}

// Sixteen bytes a lane from memory into LDS, the lanes' pieces one behind the other from `to` on. The s_nop is the wait state
// between writing m0 and the load.
static __device__ __forceinline__ void load_to_lds(const void* from, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(from) : "m0");
}

// The same from `from` + lane_at + wave_at, `from` as `buffer_of` describes it.
static __device__ __forceinline__ void buffer_to_lds(const intx4& from, int lane_at, int wave_at, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(lane_at), "s"(from),
               "s"(wave_at)
               : "m0");
}

// A buffer of `bytes` from `base` on (both the same in all lanes): reads beyond it give zeros.
static __device__ __forceinline__ intx4 buffer_of(const void* base, uint32_t bytes) {
  const uint64_t at = reinterpret_cast<uint64_t>(base);
  intx4 d;
  d[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(at));
  d[1] = __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32) & 0xffff);
  d[2] = __builtin_amdgcn_readfirstlane(static_cast<int>(bytes));
  d[3] = 0x00020000;
  return d;
}

// All but the newest LEFT loads into LDS of this wave have arrived and what it read from LDS is in its registers; then the
// same for all waves.
template <int LEFT>
static __device__ __forceinline__ void lds_arrived() {
  static_assert(LEFT < 64, "the counter's range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
