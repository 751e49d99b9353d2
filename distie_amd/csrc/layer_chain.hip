// What a decode step of few rows does between two layers' attention, in one launch: the output projection with the residual sum,
// the norm, the gated product, the down product with its residual sum, and, where another layer follows, that layer's norm and
// its q/k/v product with bias, rotation and cache write (worker/src/inference/qwen2/model.py:85-117, 149-152, 228-240, 279-290).
//
// Kernel by kernel these are six launches of 4 to 12 us, each a chain of its own: launch, a trip to memory for x, the weights
// behind it. Here a phase's first weights are on their way while the phase before still hands its results round. 1.5B shape (C 1,536,
// 93 MB of weights a layer, every layer's from memory), us a layer, this / six kernels: 1 row 25.9 / 36.8, 2 rows 26.8 / 37.2, 4 rows
// 29.5 / 37.9, 8 rows 33.0 / 39.4. What bounds it now: the weights at 5.3 TB/s while they stream (17 us), and per phase a store, the
// trip of whoever reads it, and at most 1 us of products and sums.
//
// One workgroup a compute unit, all of them work on every phase. A phase's product is cut into units (a block of 16 rows of W with its
// whole K; half a block, eight rows, for the sums, so that 1,536 rows occupy 192 units), units into `slots`, one a workgroup. In a
// workgroup eight waves stream weights (each an eighth of K, from memory straight into a ring of its own in LDS, which holds what the
// wave asks for ahead) and four others do the rest: x in front of the product, the sum of the eight waves' parts and its end behind it. A
// wave's loads return in the order of issue, so a wave that polls must have no weights under way; and a compute unit's loads queue, so
// the next weights are asked for only behind the stores that others wait for (asked for before them: 3.2 us a layer more with 1 row, 14
// with 8). Weights are loaded past the caches (`nt`: 1.3 us a layer less). Asking for less ahead: 27.2 and 28.5 us with four and two
// groups of the ring's six.
//
// Values go from workgroup to workgroup through memory, and each 32-bit word says by itself whether it is there: the buffers (`mid`,
// `hidden`, `out`) hold UNWRITTEN everywhere when the launch begins, nobody writes that pattern (a NaN; `written`), words are stored and
// loaded past the caches that workgroups do not share (stores and loads at device scope), and a reader repeats its loads until no word is
// missing. So no order between two words, no acknowledgement, counter or fence is needed. With counters (store, acknowledgement,
// count, poll, load) each boundary cost five trips instead of two, and the layer at 1 row 14 us more than now.
//
// Nothing here waits for a workgroup that has not started. A workgroup claims its slot of every phase when it starts; one that finds its x
// incomplete for `patience` looks takes, of the earliest phase that has any, a slot that nobody has claimed, works on it as on its own,
// and then goes on. The earliest phase that is not complete consists of slots claimed by running workgroups, whose x is complete, and of
// unclaimed ones, which the first to lose its patience takes: some workgroup always gets on, whatever else runs on the device.
// (`limit` rounds of that without an end are never reached; a workgroup that reached them would write NaN, say so in `gave_up`, which
// the host reads with the step's result, and leave.)
#include "lds_load.h"
#include "packed.h"
#include <algorithm>

namespace {

constexpr int STREAM = 8;                 // waves that stream weights
constexpr int HELP = 4;                   // waves in front of and behind the products
constexpr int MAX_PHASES = 4;
constexpr int ROWS = 8;                   // rows of x at most
constexpr int TILE = PK_TILE * 2;         // bytes of a tile of the packed copy
constexpr int XPAD = 8;                   // elements between the rows of x in LDS
constexpr int JOB = 128;                  // bytes in front of the parts of LDS
constexpr int OUTSIDE = 0x40000000;       // beyond every buffer: read as zeros
constexpr uint32_t UNWRITTEN = 0xffffffffu;

enum { KIND_SUM = 0, KIND_GATED = 1, KIND_ROTARY = 2 };

struct Phase {
  const bf16_t* w;                        // packed copy
  const bf16_t* x;                        // KIND_SUM: [M, K]
  const float* norm_weight;               // the others: [C], of the norm of `from` in front of the product
  const float* from;                      // [M, C]: what is normed, or what a sum is added to
  void* to;
  float eps;
  int kind, tiles;                        // tiles of K
  int slots, each, extra;                 // slots with units: the first `extra` hold each + 1 of them, the others `each`
};

struct Chain {
  Phase phase[MAX_PHASES];
  const float* bias;
  RotaryOut rotary;
  int32_t* claims;                        // [phase][slot], UNWRITTEN: nobody's
  int32_t* gave_up;                       // in host memory: 1 once a wait came to its end without what it was for
  int M, I, NQ, phases, slots, patience, limit;
};

// The arguments, read where they are needed: kept from the start they would fill the scalar registers.
typedef const __attribute__((address_space(4))) Chain* Args;

// A barrier for what the waves hand each other through LDS: loads from memory stay under way.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// All but the newest LEFT loads of this wave have arrived.
template <int LEFT>
__device__ __forceinline__ void arrived() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}

// G tiles from `at` on, one behind the other in memory and in LDS. (The offset of an instruction counts on both sides.)
template <int G>
__device__ __forceinline__ void load_group(const intx4& from, int at, uint32_t to) {
#define FIRST "s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
#define NEXT(more) "\n\tbuffer_load_dwordx4 %1, %2, 0 offen offset:" #more " nt lds"
  static_assert(G == 3 || G == 4, "offsets of 12 bits");
  const uint32_t lds_at = __builtin_amdgcn_readfirstlane(to);
  if constexpr (G == 4)
    asm volatile(FIRST NEXT(1024) NEXT(2048) NEXT(3072) ::"s"(lds_at), "v"(at), "s"(from) : "m0");
  else
    asm volatile(FIRST NEXT(1024) NEXT(2048) ::"s"(lds_at), "v"(at), "s"(from) : "m0");
#undef FIRST
#undef NEXT
}

// Sixteen bytes of what other workgroups of the launch write, and eight for them, at device scope.
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t uintx4;
extern "C" __device__ uintx4 chain_buffer_load(intx4 from, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.v4i32");
constexpr int DEVICE_SCOPE = 16;          // sc1
__device__ __forceinline__ uintx4 load_shared(const intx4& from, int at) { return chain_buffer_load(from, at, 0, DEVICE_SCOPE); }
// In front of every look for what may not be there yet. The load is declared to read memory and do nothing else: a loop that does not
// say that memory changes could be given the first look's answer for ever.
__device__ __forceinline__ void look_again() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ bool unwritten(const uintx4& v) {
  return v[0] == UNWRITTEN || v[1] == UNWRITTEN || v[2] == UNWRITTEN || v[3] == UNWRITTEN;
}
__device__ __forceinline__ uint32_t written(uint32_t v) { return v == UNWRITTEN ? 0x7fc07fc0u : v; }   // a NaN either way
__device__ __forceinline__ void store_shared(void* p, uint32_t a, uint32_t b) {
  __hip_atomic_store(static_cast<uint64_t*>(p), static_cast<uint64_t>(written(a)) | (static_cast<uint64_t>(written(b)) << 32),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void give_up(int32_t* flag) { __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }

// T: tiles of C a wave; G: tiles of a group, which are asked for together; R: groups of a wave's ring; B: groups of x a wave keeps (sums)
template <int T, int G, int R, int B>
__global__ __launch_bounds__(64 * (STREAM + HELP)) __attribute__((amdgpu_waves_per_eu(3, 3)))
void layer_chain_kernel(const Chain given) {
  Args args = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int C = T * 256;
  constexpr int XK = C + XPAD;
  constexpr int RING = R * G * TILE;
  extern __shared__ char chain_lds[];
  // [1]: the phases whose slot is this workgroup's; [0]: someone found x incomplete; [2]: how deep, behind that, the jobs of
  // others lie in [4 ..] (phase, slot), one below the other
  int* const job = reinterpret_cast<int*>(chain_lds);
  char* const rings = chain_lds + JOB;
  bf16_t* const xs = reinterpret_cast<bf16_t*>(rings + STREAM * RING);                       // [M][XK]
  floatx4* const part = reinterpret_cast<floatx4*>(rings + STREAM * RING + args->M * XK * 2);       // [unit][wave][4][M]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lane = threadIdx.x % 64;
  const int own = blockIdx.x;
  const int M = args->M;

  if (wave < STREAM) {
    // ---- the waves that stream
    const char* const ring = rings + wave * RING;
    const uint32_t ring_at = lds_place(ring);
    const int r = lane % 16, g = lane / 16;
    // A sum's operand holds eight rows of W twice, the second time G tiles further on, and x accordingly: what the matrix product
    // has on its diagonal blocks of 8 x 8 are two parts of the sum.
    const int half_at = (r / 8) * (G * TILE) + (16 * g + r % 8) * 16;
    const int part_at = r < M ? M * g + r : -1;
    const int part_sum = (r < 8) == (g < 2) && r % 8 < M ? M * g + r % 8 : -1;
    // what is asked for next: group `at` of [first, last) of unit `unit`, into place `ring_group`
    const bf16_t *weights, *block;
    int kind, tiles, unit, units, first, last, at, wave_at, lane_at, ring_group;
    int asked_p = -1, asked_s = -1;
    auto start_unit = [&]() __attribute__((always_inline)) {
      const bool sum = kind == KIND_SUM;
      block = weights + static_cast<int64_t>(sum ? unit / 2 : unit) * tiles * PK_TILE;
      lane_at = sum ? half_at + (unit % 2) * 128 : lane * 16;
      wave_at = first * (sum ? 2 * G * TILE : G * TILE);
      at = first;
    };
    auto ask = [&]() __attribute__((always_inline)) {
      if (units > 0) {
        // (beyond the block: zeros, where K is no multiple of a sum's groups)
        load_group<G>(buffer_of(block, tiles * TILE), lane_at + wave_at, ring_at + ring_group * (G * TILE));
        wave_at += kind == KIND_SUM ? 2 * G * TILE : G * TILE;
        ring_group = ring_group + 1 == R ? 0 : ring_group + 1;
        if (++at == last) {
          --units;
          ++unit;
          start_unit();
        }
      }
    };
    auto begin = [&](int p, int slot) __attribute__((always_inline)) {       // nothing of the wave's is under way
      Args now = args;
      asm volatile("" : "+s"(now));
      kind = now->phase[p].kind;
      tiles = now->phase[p].tiles;
      weights = now->phase[p].w;
      unit = slot * now->phase[p].each + min(slot, now->phase[p].extra);
      units = now->phase[p].each + (slot < now->phase[p].extra);
      if (kind == KIND_SUM) {
        const int groups = (tiles + 2 * G - 1) / (2 * G);
        first = wave * groups / STREAM;
        last = (wave + 1) * groups / STREAM;
        if (first == last) units = 0;
      } else {
        first = wave * (T / G);
        last = first + T / G;
      }
      ring_group = 0;
      asked_p = p;
      asked_s = slot;
      start_unit();
#pragma unroll
      for (int e = 0; e < R; ++e) ask();
    };
    int p = 0, depth = 0, q = 0, slot = own, owned = -1;
    bool known = false;                                          // `owned` is; the first weights are asked for in any case
    while (p < args->phases) {
      if (depth == 0) {
        q = p;
        slot = own;
        if (!((owned >> p) & 1) || own >= args->phase[p].slots) {
          ++p;
          continue;
        }
      } else {
        q = __builtin_amdgcn_readfirstlane(job[4 + 2 * depth]);
        slot = __builtin_amdgcn_readfirstlane(job[5 + 2 * depth]);
      }
      if (q != asked_p || slot != asked_s) {
        arrived<0>();                                            // what was asked for is not for this job
        begin(q, slot);
      }
      if (!known) {
        lds_barrier();                                           // (1)
        owned = __builtin_amdgcn_readfirstlane(job[1]);
        known = true;
        continue;
      }
      const int n = args->phase[q].each + (slot < args->phase[q].extra);
      int left = 0;                                              // groups that are still to be multiplied
      int group = 0;                                             // place of the next one
      bf16x8 w[G];
      auto take = [&]() __attribute__((always_inline)) {
        if (left >= R) arrived<(R - 1) * G>(); else arrived<0>();
        const char* from = ring + group * (G * TILE) + lane * 16;
#pragma unroll
        for (int e = 0; e < G; ++e) w[e] = *reinterpret_cast<const bf16x8*>(from + e * TILE);
        group = group + 1 == R ? 0 : group + 1;
        --left;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // its place is free again
        ask();
      };
      // x is there, or someone found it incomplete: then a job of an earlier phase may come first
      auto late = [&]() __attribute__((always_inline)) -> bool {
        lds_barrier();                                           // (2)
        if (!__builtin_amdgcn_readfirstlane(job[0])) return false;
        lds_barrier();                                           // (3)
        lds_barrier();                                           // (4)
        depth = __builtin_amdgcn_readfirstlane(job[2]);
        return true;
      };
      floatx4* flush = part + wave * 4 * M;
      if (args->phase[q].kind == KIND_SUM) {
        const int all = args->phase[q].tiles, groups = (all + 2 * G - 1) / (2 * G);
        const int begins = wave * groups / STREAM, run = (wave + 1) * groups / STREAM - begins;
        const intx4 from = buffer_of(args->phase[q].x, M * all * 64);
        const int t0 = begins * (2 * G) + (r / 8) * G;
        const int x_at = (min(r % 8, M - 1) * (all * 4) + g) * 16 + t0 * 64;
        uintx4 x[B][G];
        int tries = args->patience;
        for (;;) {
          look_again();
          bool missing = false;
#pragma unroll
          for (int b = 0; b < B; ++b) {
            const int b_at = x_at + (b < run ? 2 * G * b * 64 : OUTSIDE);
#pragma unroll
            for (int e = 0; e < G; ++e) x[b][e] = load_shared(from, b_at + e * 64);
          }
#pragma unroll
          for (int b = 0; b < B; ++b)
#pragma unroll
            for (int e = 0; e < G; ++e) missing |= unwritten(x[b][e]);
          if (q == 0 || !__any(missing)) break;                  // (the first phase's x is an argument of the launch)
          if (--tries <= 0) {
            if (lane == 0) job[0] = 1;
            break;
          }
        }
        if (2 * G * (begins + run) > all) {                      // the last group reaches beyond K, into the next row of x
#pragma unroll
          for (int b = 0; b < B; ++b)
#pragma unroll
            for (int e = 0; e < G; ++e) {
              const bool in = t0 + 2 * G * b + e < all;
#pragma unroll
              for (int i = 0; i < 4; ++i) x[b][e][i] = in ? x[b][e][i] : 0u;
            }
        }
        if (late()) {
          if (depth < 0) { arrived<0>(); return; }
          continue;
        }
        left = n * run;
        for (int u = 0; u < n; ++u) {
          floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int b = 0; b < B; ++b) {
            if (b < run) {
              take();
#pragma unroll
              for (int e = 0; e < G; ++e)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[e], __builtin_bit_cast(bf16x8, x[b][e]), acc, 0, 0, 0);
            }
          }
          if (part_sum >= 0) flush[part_sum] = acc;
          flush += STREAM * 4 * M;
        }
      } else {
        if (late()) {
          if (depth < 0) { arrived<0>(); return; }
          continue;
        }
        left = n * (T / G);
        const bf16_t* const xp = xs + min(r, M - 1) * XK + 8 * g + 32 * T * wave;
        bf16x8 x[T];
#pragma unroll
        for (int e = 0; e < T; ++e) x[e] = *reinterpret_cast<const bf16x8*>(xp + 32 * e);
        while (left > 0) {
          floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int h = 0; h < T / G; ++h) {
            take();
#pragma unroll
            for (int e = 0; e < G; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[e], x[h * G + e], acc, 0, 0, 0);
          }
          if (part_at >= 0) flush[part_at] = acc;
          flush += STREAM * 4 * M;
        }
      }
      lds_barrier();                                             // (5): the parts of the sums are in LDS
      lds_barrier();                                             // (6): the results are on their way
      asked_p = -1;
      if (depth > 0)
        --depth;
      else
        ++p;
    }
    if (!known) lds_barrier();                                   // (1)
    arrived<0>();
    return;
  }

  // ---- the waves that help
  __builtin_amdgcn_s_setprio(3);
  const int helper = wave - STREAM;
  const int r = lane % 8, g = lane / 8 % 2;                      // of a unit's sums: token r, rows 4 g .. + 3
  if (helper == 0) {
    int mine = 0;
    if (lane < args->phases && own < args->phase[lane].slots)
      mine = __hip_atomic_exchange(args->claims + lane * args->slots + own, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             static_cast<int32_t>(UNWRITTEN);
    const uint64_t mask = __ballot(mine);
    if (lane == 0) {
      job[0] = 0;
      job[1] = static_cast<int>(mask);
    }
  }
  lds_barrier();                                                 // (1)
  if (helper == HELP - 1) {
    // every line of the arguments once, so that what is read of them later is in the scalar cache
    const __attribute__((address_space(4))) int* word = (const __attribute__((address_space(4))) int*)args;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(Chain) / 4); i += 16) sum += word[i];
    asm volatile("" ::"s"(sum));
  }
  const int owned = __builtin_amdgcn_readfirstlane(job[1]);
  int p = 0, depth = 0, rounds = 0, q = 0, slot = own;
  while (p < args->phases) {
    if (depth == 0) {
      q = p;
      slot = own;
      if (!((owned >> p) & 1)) {
        ++p;
        continue;
      }
    } else {
      q = __builtin_amdgcn_readfirstlane(job[4 + 2 * depth]);
      slot = __builtin_amdgcn_readfirstlane(job[5 + 2 * depth]);
    }
    const int kind = args->phase[q].kind;
    const int each = args->phase[q].each, extra = args->phase[q].extra;
    const int u0 = slot * each + min(slot, extra), n = each + (slot < extra);
    const intx4 from = buffer_of(args->phase[q].from, M * C * 4);
    if (kind != KIND_SUM) {
      // rows `helper`, helper + HELP, .. of the residual sum, until they are complete; then their norm
      float4 nw[T];
      const float* const weight = args->phase[q].norm_weight;
#pragma unroll
      for (int e = 0; e < T; ++e) nw[e] = *reinterpret_cast<const float4*>(weight + 4 * lane + 256 * e);
      const float eps = args->phase[q].eps;
      uintx4 v[ROWS / HELP][T];
      int tries = args->patience;
      bool missing;
      do {
        look_again();
#pragma unroll
        for (int i = 0; i < ROWS / HELP; ++i) {
          const int m = helper + HELP * i, at = (m < M ? m * C * 4 : OUTSIDE) + 16 * lane;
#pragma unroll
          for (int e = 0; e < T; ++e) v[i][e] = load_shared(from, at + 1024 * e);
        }
        missing = false;
#pragma unroll
        for (int i = 0; i < ROWS / HELP; ++i)
#pragma unroll
          for (int e = 0; e < T; ++e) missing |= unwritten(v[i][e]);
      } while (__any(missing) && --tries > 0);
      if (tries <= 0 && lane == 0) job[0] = 1;
#pragma unroll
      for (int i = 0; i < ROWS / HELP; ++i) {
        const int m = helper + HELP * i;
        if (m < M) {
          // (vectors are cast whole: the cast of an element gave element 0 for each of them)
          float ss = 0.f;
#pragma unroll
          for (int e = 0; e < T; ++e) {
            const float4 f = __builtin_bit_cast(float4, v[i][e]);
            ss += f.x * f.x + f.y * f.y + f.z * f.z + f.w * f.w;
          }
          const float scale = rsqrtf(wave_sum(ss) / static_cast<float>(C) + eps);
#pragma unroll
          for (int e = 0; e < T; ++e) {
            const float4 f = __builtin_bit_cast(float4, v[i][e]);
            const float o[4] = {f.x * scale * nw[e].x, f.y * scale * nw[e].y, f.z * scale * nw[e].z, f.w * scale * nw[e].w};
            *reinterpret_cast<uint2*>(xs + m * XK + 4 * lane + 256 * e) = pack_bf16x4(o);
          }
        }
      }
    }
    lds_barrier();                                               // (2): x is there, or someone found it incomplete
    if (__builtin_amdgcn_readfirstlane(job[0])) {
      lds_barrier();                                             // (3)
      if (helper == 0) {
        int found_p = -1, found_s = -1;
        for (int e = 0; e < q && found_p < 0; ++e) {
          const int slots = args->phase[e].slots;
          int32_t* const claims = args->claims + e * args->slots;
          for (int s0 = 0; s0 < slots && found_p < 0; s0 += 64) {
            const int s = s0 + lane;
            const int32_t taken = s < slots ? __hip_atomic_load(claims + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 1;
            const uint64_t open = __ballot(taken == static_cast<int32_t>(UNWRITTEN));
            if (open) {
              const int free = s0 + __builtin_ctzll(open);
              int32_t before = 1;
              if (lane == 0) before = __hip_atomic_exchange(claims + free, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              if (__builtin_amdgcn_readfirstlane(before) == static_cast<int32_t>(UNWRITTEN)) {
                found_p = e;
                found_s = free;
              }
            }
          }
        }
        const bool over = ++rounds >= args->limit;
        if (lane == 0) {
          job[0] = 0;
          if (found_p >= 0) {                                    // (jobs below one another are of falling phases: four at most)
            job[4 + 2 * (depth + 1)] = found_p;
            job[5 + 2 * (depth + 1)] = found_s;
          }
          job[2] = over ? -1 : depth + (found_p >= 0);
        }
      }
      lds_barrier();                                             // (4): job[2]: deeper, the same again, or given up
      depth = __builtin_amdgcn_readfirstlane(job[2]);
      if (depth < 0) {
        if (helper == 0 && lane == 0) give_up(args->gave_up);
        if (helper == 0)
          for (int i = lane; i < M * 8; i += 64)
            if (8 * own < C) static_cast<float*>(args->phase[2].to)[(i / 8) * C + 8 * own + i % 8] = __builtin_nanf("");
        return;
      }
      continue;
    }
    // What a sum is added to, asked for while the product is under way. It was complete before x was, since whoever wrote x had
    // read all of it: the first look finds it. (A word that `limit` looks did not find is added as the NaN that it holds.)
    void* const to = args->phase[q].to;
    auto added_to = [&](int at) __attribute__((always_inline)) {
      uintx4 v;
      int tries = args->limit;
      do {
        look_again();
        v = load_shared(from, at);
      } while (q > 0 && unwritten(v) && --tries > 0);
      if (tries == 0) give_up(args->gave_up);
      return v;
    };
    uintx4 old = {};
    int k = helper * 4 + lane / 16;
    if (kind == KIND_SUM && k < n && r < M) old = added_to((r * C + 8 * (u0 + k) + 4 * g) * 4);
    lds_barrier();                                               // (5): the parts of the sums are in LDS
    for (; k < n; k += HELP * 4) {
      const int u = u0 + k;
      if (r < M) {
        // rows 4 g .. + 3 of the block and the four that lie eight rows further on, over the waves
        const floatx4* sums = part + (k * STREAM * 4 + g) * M + r;
        float near[4] = {}, far[4] = {};
#pragma unroll 1
        for (int v = 0; v < STREAM; v += 4) {
          floatx4 t[4][2];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) t[i][h] = sums[(4 * (v + i) + 2 * h) * M];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            near[i] += (t[0][0][i] + t[1][0][i]) + (t[2][0][i] + t[3][0][i]);
            far[i] += (t[0][1][i] + t[1][1][i]) + (t[2][1][i] + t[3][1][i]);
          }
        }
        if (kind == KIND_SUM) {
          const int at = r * C + 8 * u + 4 * g;
          if (k >= HELP * 4) old = added_to(at * 4);
          const float4 sum = __builtin_bit_cast(float4, old);
          store_shared(static_cast<float*>(to) + at, __builtin_bit_cast(uint32_t, sum.x + (near[0] + far[0])),
                       __builtin_bit_cast(uint32_t, sum.y + (near[1] + far[1])));
          store_shared(static_cast<float*>(to) + at + 2, __builtin_bit_cast(uint32_t, sum.z + (near[2] + far[2])),
                       __builtin_bit_cast(uint32_t, sum.w + (near[3] + far[3])));
        } else if (kind == KIND_GATED) {
          float h[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) h[i] = gate_activation(near[i], 0) * far[i];
          const uint2 v = pack_bf16x4(h);
          store_shared(static_cast<bf16_t*>(to) + r * args->I + 8 * u + 4 * g, v.x, v.y);
        } else {
          // block (head, sub): of a q or k head its rows 8 sub .. + 7 and those half a head further on, of a v head 16 in order
          const int dim = args->rotary.dim, half = dim / 2, per_head = dim / 16;
          const int head = u / per_head, sub = u % per_head, heads = args->rotary.heads, turned = heads + args->rotary.kv_heads;
          const bool turns = head < turned;
          const int d0 = (turns ? 8 : 16) * sub + 4 * g, d1 = d0 + (turns ? half : 8);
          const float* const bias = args->bias;
          const int place = args->rotary.write ? args->rotary.slots[r] : 0;
          float a[4], b[4], lo[4], hi[4];
          float2 cs[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            cs[i] = turns ? args->rotary.table[r * half + d0 + i] : float2{1.f, 0.f};
            a[i] = near[i] + (bias != nullptr ? bias[head * dim + d0 + i] : 0.f);
            b[i] = far[i] + (bias != nullptr ? bias[head * dim + d1 + i] : 0.f);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            lo[i] = turns ? a[i] * cs[i].x - b[i] * cs[i].y : a[i];
            hi[i] = turns ? b[i] * cs[i].x + a[i] * cs[i].y : b[i];
          }
          const uint2 lo4 = pack_bf16x4(lo), hi4 = pack_bf16x4(hi);
          bf16_t* const row = static_cast<bf16_t*>(to) + r * args->NQ + head * dim;
          *reinterpret_cast<uint2*>(row + d0) = lo4;
          *reinterpret_cast<uint2*>(row + d1) = hi4;
          if (args->rotary.write && head >= heads) {
            const int block = args->rotary.block_size;
            const int64_t page = place / block;
            const int offset = place % block;
            if (turns) {
              bf16_t* const key = args->rotary.k_cache + ((page * args->rotary.kv_heads + (head - heads)) * block + offset) * dim;
              *reinterpret_cast<uint2*>(key + d0) = lo4;
              *reinterpret_cast<uint2*>(key + d1) = hi4;
            } else {
              bf16_t* const value = args->rotary.v_cache + (page * args->rotary.kv_heads + (head - turned)) * dim * block + offset;
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                value[static_cast<int64_t>(d0 + i) * block] = static_cast<bf16_t>(lo[i]);
                value[static_cast<int64_t>(d1 + i) * block] = static_cast<bf16_t>(hi[i]);
              }
            }
          }
        }
      }
    }
    lds_barrier();                                               // (6): the results are on their way
    if (depth > 0)
      --depth;
    else
      ++p;
  }
}

constexpr int LDS_BYTES = 160 * 1024;

// Groups of a wave's ring, as many as LDS has room for beside up to 2 rows of x, and beside up to ROWS: 4 rows in rings of six and of
// four groups of three tiles 30.7 / 30.0 us a layer, 1 row 27.2 / 28.3 (both before the weights went past the caches).
int ring_bytes(int C, int M) {
  const bool few = M <= 2;
  return STREAM * TILE * (C == 1024 ? (few ? 16 : 12) : C == 1536 ? (few ? 18 : 12) : (few ? 16 : 12));
}

int lds_bytes(int M, int C, int most) { return JOB + ring_bytes(C, M) + M * (C + XPAD) * 2 + most * STREAM * M * 64; }

int most_units(int units, int slots) { return (units + slots - 1) / slots; }

// The longest K of a sum: its x stays in the registers of eight waves.
int longest(int C) { return C == 1024 ? STREAM * 4 * 8 * 32 : C == 1536 ? STREAM * 6 * 6 * 32 : C == 2048 ? STREAM * 6 * 8 * 32 : 0; }

template <int T, int G, int R, int B>
int launch(const Chain& a, int grid, int bytes, hipStream_t stream) {
  layer_chain_kernel<T, G, R, B><<<grid, 64 * (STREAM + HELP), bytes, stream>>>(a);
  return launch_status();
}

}  // namespace

// Whether these sizes run here: x [M, ..], residual [M, C], attention's result [M, KO], I hidden values, NQ columns of q, k and v
// behind it (0: none); `slots`: compute units.
extern "C" int distie_layer_chain_fits(int M, int C, int KO, int I, int NQ, int slots) {
  if (M < 1 || M > ROWS || KO % 32 || I % 32 || KO < 32 || I < 32 || KO > longest(C) || I > longest(C) || NQ % 16 || NQ < 0 ||
      NQ > 65536 || slots < 1 || slots > 1024)
    return 0;
  const int most = std::max(std::max(most_units(C / 8, slots), most_units(I / 8, slots)), most_units(NQ / 16, slots));
  return lds_bytes(M, C, most) <= LDS_BYTES;
}

// 32-bit words of `claims`
extern "C" int distie_layer_chain_claims(int slots) { return MAX_PHASES * slots; }

// mid, out: float32 [M, C], hidden: bfloat16 [M, I], claims: all of them UNWRITTEN (bytes of 0xff) when the launch begins, each at a
// multiple of 16 bytes. qkv_w null: no layer follows. grid: workgroups (`slots`. With fewer, to try what they do for others, the
// last phase keeps its holes: nobody waits for it, it is left to those who start late). gave_up: host memory that the device writes.
extern "C" int distie_layer_chain(const void* mixed, const void* o_w, const float* residual, float* mid, const float* norm, float eps,
                                  const void* gate_up_w, void* hidden, const void* down_w, float* out, const float* next_norm,
                                  float next_eps, const void* qkv_w, const float* bias, void* qkv, const void* table,
                                  const int32_t* cache_slots, void* k_cache, void* v_cache, int heads, int kv_heads, int dim,
                                  int block_size, int write, int M, int C, int KO, int I, int32_t* claims, int32_t* gave_up, int slots,
                                  int grid, int patience, int limit, hipStream_t stream) {
  const int NQ = qkv_w != nullptr ? (heads + 2 * kv_heads) * dim : 0;
  if (!distie_layer_chain_fits(M, C, KO, I, NQ, slots) || grid < 1 || grid > slots || patience < 1 || limit < 1 ||
      gave_up == nullptr)
    return DISTIE_BAD_ARGUMENT;
  if (qkv_w != nullptr && (heads < 1 || kv_heads < 1 || dim < 16 || dim % 16 || block_size < 1)) return DISTIE_BAD_ARGUMENT;
  Chain a = {};
  a.phases = qkv_w != nullptr ? 4 : 3;
  const void* weights[MAX_PHASES] = {o_w, gate_up_w, down_w, qkv_w};
  const void* xs[MAX_PHASES] = {mixed, nullptr, hidden, nullptr};
  const float* norms[MAX_PHASES] = {nullptr, norm, nullptr, next_norm};
  const float* from[MAX_PHASES] = {residual, mid, mid, out};
  void* to[MAX_PHASES] = {mid, hidden, out, qkv};
  const int kinds[MAX_PHASES] = {KIND_SUM, KIND_GATED, KIND_SUM, KIND_ROTARY};
  const int K[MAX_PHASES] = {KO, C, I, C}, units[MAX_PHASES] = {C / 8, I / 8, C / 8, NQ / 16};
  for (int p = 0; p < a.phases; ++p) {
    Phase& f = a.phase[p];
    f.w = static_cast<const bf16_t*>(weights[p]);
    f.x = static_cast<const bf16_t*>(xs[p]);
    f.norm_weight = norms[p];
    f.eps = p == 1 ? eps : next_eps;
    f.from = from[p];
    f.to = to[p];
    f.kind = kinds[p];
    f.tiles = K[p] / 32;
    f.slots = std::min(slots, units[p]);
    f.each = units[p] / f.slots;
    f.extra = units[p] % f.slots;
  }
  a.bias = bias;
  a.rotary = RotaryOut{static_cast<const float2*>(table), cache_slots, static_cast<bf16_t*>(k_cache), static_cast<bf16_t*>(v_cache),
                       heads, kv_heads, dim, block_size, write, 0, 0.f, 1.f, 0.f};
  a.claims = claims;
  a.gave_up = gave_up;
  a.M = M;
  a.I = I;
  a.NQ = NQ;
  a.slots = slots;
  a.patience = patience;
  a.limit = limit;
  const int most = std::max(std::max(most_units(C / 8, slots), most_units(I / 8, slots)), most_units(NQ / 16, slots));
  const int bytes = lds_bytes(M, C, most);
  switch (C) {
    case 1024: return M <= 2 ? launch<4, 4, 4, 4>(a, grid, bytes, stream) : launch<4, 4, 3, 4>(a, grid, bytes, stream);
    case 1536: return M <= 2 ? launch<6, 3, 6, 6>(a, grid, bytes, stream) : launch<6, 3, 4, 6>(a, grid, bytes, stream);
    case 2048: return M <= 2 ? launch<8, 4, 4, 6>(a, grid, bytes, stream) : launch<8, 4, 3, 6>(a, grid, bytes, stream);
  }
  return DISTIE_BAD_ARGUMENT;
}
