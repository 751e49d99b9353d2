// Attention over the paged cache for one head size (compile with -DDISTIE_HEAD_DIM=<even size up to 1024>; the
// matrix-core kernels exist for multiples of 16 only, the wave-per-token kernel for every even size).
//
// out[t, h] = softmax_j(q[t, h] . k[j, h / G] * scale) v[j, h / G] over the keys j that token t may see:
// first(t) <= j <= position(t): first = 0 (window 0), position - window + 1 (window > 0), or the start of the run of
// -window positions that the token lies in, counted from position 0 (window < 0: chunks that see only themselves). Keys and values
// are read through the block table of the token's request (row table_rows[request] of block_table, or row
// `request` itself when table_rows is null): key j lives in page table[j / P] at offset
// j % P of a cache laid out k [pages, kv_heads, P, D], v [pages, kv_heads, D, P]. The new tokens of the step are
// already in the cache
// (the reference writes before it reads too: worker/src/inference/qwen2/paged_attn.py:389-397), so
// prefill, portions of prompts and decoded tokens are the same computation.
// Formula: worker/src/inference/qwen2/model.py:154-161; softmax and all sums in float32.
//
//  * attn_generic: one wave per (token, head); any types; the true 32-bit path and the fallback.
//  * attn_decode + attn_reduce, attn_prefill, attn_prefill_keys: bfloat16 on the matrix cores (described further down).

#include "common.h"
#include "lds_load.h"
#include <algorithm>

#ifndef DISTIE_HEAD_DIM
#error "compile with -DDISTIE_HEAD_DIM=<head size>"
#endif
#if DISTIE_HEAD_DIM % 2 != 0 || DISTIE_HEAD_DIM < 2 || DISTIE_HEAD_DIM > 1024
#error "head size must be even and at most 1024"
#endif
// (beyond 256 the matrix-core kernels' tiles no longer fit their registers and LDS: the wave-per-token kernel serves)
#define DISTIE_MATRIX_CORE_ATTENTION (DISTIE_HEAD_DIM % 16 == 0 && DISTIE_HEAD_DIM <= 256)

constexpr int D = DISTIE_HEAD_DIM;
constexpr int DIMS_PER_LANE = (D + DISTIE_WAVE - 1) / DISTIE_WAVE;

extern "C" int distie_attention_head_dim() { return D; }

// the first key that the token at position `pos` sees (`window`: see above; never falls as the position grows)
__device__ __forceinline__ int first_visible(int pos, int window) {
  if (window > 0) return max(0, pos - window + 1);
  return window < 0 ? pos - pos % -window : 0;
}

template <typename C>
__device__ __forceinline__ float dot_row(const float* q, const C* k);

template <>
__device__ __forceinline__ float dot_row<float>(const float* q, const float* k) {
  float s = 0.f;
  if constexpr (D % 4 != 0) {                  // rows are not 16-byte aligned: element by element
#pragma unroll
    for (int d = 0; d < D; ++d) s = fmaf(q[d], k[d], s);
    return s;
  }
#pragma unroll
  for (int d = 0; d + 4 <= D; d += 4) {
    const float4 v = *reinterpret_cast<const float4*>(k + d);
    s = fmaf(q[d], v.x, s);
    s = fmaf(q[d + 1], v.y, s);
    s = fmaf(q[d + 2], v.z, s);
    s = fmaf(q[d + 3], v.w, s);
  }
  return s;
}

template <>
__device__ __forceinline__ float dot_row<bf16_t>(const float* q, const bf16_t* k) {
  float s = 0.f;
  if constexpr (D % 8 != 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) s = fmaf(q[d], to_float(k[d]), s);
    return s;
  }
#pragma unroll
  for (int d = 0; d + 8 <= D; d += 8) {
    const uint4 raw = *reinterpret_cast<const uint4*>(k + d);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s = fmaf(q[d + 2 * i], __uint_as_float(w[i] << 16), s);
      s = fmaf(q[d + 2 * i + 1], __uint_as_float(w[i] & 0xffff0000u), s);
    }
  }
  return s;
}

// four consecutive values of a page's row of V^T as floats
__device__ __forceinline__ void load4(const float* p, float v[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float v[4]) {
  const uint2 raw = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(raw.x << 16); v[1] = __uint_as_float(raw.x & 0xffff0000u);
  v[2] = __uint_as_float(raw.y << 16); v[3] = __uint_as_float(raw.y & 0xffff0000u);
}

// The sums over lanes of attn_generic_kernel. In the vector ALU only where that does not take registers away from waves: with it the
// compiler has more loads under way, and heads of 96, 128 and 288 in bfloat16 went from 103 .. 118 registers to 132 .. 149, from four waves a
// SIMD to three: 100 requests of 500 keys, 32 heads of 128 on one with a bias by distance, us, through the LDS unit / in the vector ALU
// 118 / 202, of 288 261 / 450, 300 tokens of 12 heads of 96 on 2 53.2 / 60.5. Heads of 64 in bfloat16 take fewer with it (135 / 116; 0.86 of
// the time on average), in float32 107 / 91 and up to 1.10 of the time; of 16 and 40 0.97 in both.
template <typename C>
constexpr bool GENERIC_SUMS_IN_VALU = D <= (sizeof(C) == 2 ? 64 : 48);
template <typename C>
__device__ __forceinline__ float generic_sum(float v) {
  if constexpr (GENERIC_SUMS_IN_VALU<C>) return wave_sum(v);
#pragma unroll
  for (int o = DISTIE_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, DISTIE_WAVE);
  return v;
}
template <typename C>
__device__ __forceinline__ float generic_max(float v) {
  if constexpr (GENERIC_SUMS_IN_VALU<C>) return wave_max(v);
#pragma unroll
  for (int o = DISTIE_WAVE / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, DISTIE_WAVE));
  return v;
}

// One workgroup of WAVES waves per (token, head). The keys are taken in chunks of 64 that begin at multiples of
// 64; the chunks are dealt to the waves in turn (a token that decodes over thousands of keys then has eight
// waves at work instead of one), every wave keeps its own running maximum, sum and output, and wave 0 puts them
// together at the end, in wave order. In a chunk a lane owns one key for the scores; for the output it owns
// the dimensions lane, lane + 64, ... and walks the chunk's keys: a page at a time with 16-byte loads of the
// page's row of V^T when pages divide 64 and hold a multiple of four tokens, else key by key.
template <typename T, typename C, int WAVES>
__global__ __launch_bounds__(DISTIE_WAVE * WAVES) void attn_generic_kernel(
    const T* __restrict__ qkv, int64_t q_stride, const C* __restrict__ k_cache, const C* __restrict__ v_cache,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ token_request,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows, T* __restrict__ out, int heads, int kv_heads,
    int block_size, float scale, int window, const float* __restrict__ head_slopes, float score_cap,
    const float* __restrict__ sinks) {
  __shared__ float q_s[D];
  __shared__ float p_s[WAVES][DISTIE_WAVE];
  __shared__ int64_t base_s[WAVES][DISTIE_WAVE];
  __shared__ float m_s[WAVES], l_s[WAVES];
  __shared__ float acc_s[WAVES][D];
  const int lane = threadIdx.x % DISTIE_WAVE;
  const int wave = threadIdx.x / DISTIE_WAVE;
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y;
  const int kh = h / (heads / kv_heads);
  const int q_pos = positions[t];
  const int request_of_token = token_request[t];
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request_of_token] : request_of_token) * table_width;
  const T* q = qkv + t * q_stride + static_cast<int64_t>(h) * D;
  for (int d = threadIdx.x; d < D; d += DISTIE_WAVE * WAVES) q_s[d] = to_float(q[d]);
  __syncthreads();

  const int first = first_visible(q_pos, window);
  const int last = q_pos;   // inclusive
  const bool by_page = block_size % 4 == 0 && DISTIE_WAVE % block_size == 0;
  const float slope = head_slopes != nullptr ? head_slopes[h] : 0.f;
  float m = -INFINITY, l = 0.f;
  float acc[DIMS_PER_LANE];
#pragma unroll
  for (int i = 0; i < DIMS_PER_LANE; ++i) acc[i] = 0.f;

  for (int c = first / DISTIE_WAVE * DISTIE_WAVE + wave * DISTIE_WAVE; c <= last; c += DISTIE_WAVE * WAVES) {
    const int key = c + lane;
    const bool valid = key >= first && key <= last;
    float s = -INFINITY;
    int64_t base = 0;
    if (valid) {
      const int page = table[key / block_size];
      base = (static_cast<int64_t>(page) * kv_heads + kh) * block_size * D;
      s = dot_row<C>(q_s, k_cache + base + static_cast<int64_t>(key % block_size) * D) * scale;
      // what a variant of attention adds to a score (both off for plain attention): a cap that bends large
      // scores, then a bias by the distance to the key with the head's own slope
      if (score_cap > 0.f) s = score_cap * tanhf(s / score_cap);
      s += slope * static_cast<float>(key - q_pos);
    }
    const float m_new = fmaxf(m, generic_max<C>(s));
    const float alpha = m_new == -INFINITY ? 0.f : expf(m - m_new);     // 0 on the first chunk with a key (m = -inf)
    const float p = valid ? expf(s - m_new) : 0.f;
    l = l * alpha + generic_sum<C>(p);
    m = m_new;
    // what the lanes of this wave hand each other goes through the wave's own rows of LDS; the wave runs its
    // LDS traffic in order, so no barrier across waves is needed, only that the compiler keeps the order
    __builtin_amdgcn_wave_barrier();
    p_s[wave][lane] = p;
    base_s[wave][lane] = base;
    __builtin_amdgcn_wave_barrier();
    const int lo = max(first - c, 0);                                   // keys lo .. hi of the chunk count
    const int hi = min(DISTIE_WAVE - 1, last - c);
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d >= D) continue;
      float a = acc[i] * alpha;
      if (by_page) {
        for (int j0 = lo / block_size * block_size; j0 <= hi; j0 += block_size) {
          // the page of keys j0 .. j0 + P - 1: its address from a key of it that counts
          const C* row = v_cache + base_s[wave][max(j0, lo)] + static_cast<int64_t>(d) * block_size;
          for (int jj = 0; jj < block_size; jj += 4) {
            float v[4];
            load4(row + jj, v);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int j = j0 + jj + e;
              if (j >= lo && j <= hi) a = fmaf(p_s[wave][j], v[e], a);    // never a value of a key that does not count
            }
          }
        }
      } else {
        for (int j = lo; j <= hi; ++j)
          a = fmaf(p_s[wave][j], to_float(v_cache[base_s[wave][j] + static_cast<int64_t>(d) * block_size + (c + j) % block_size]), a);
      }
      acc[i] = a;
    }
  }
  T* o = out + (t * heads + h) * D;
  // a sink joins the denominator as exp(sink), once, with no value: as one more maximum and one more term of the sum
  const float sink = sinks != nullptr ? sinks[h] : -INFINITY;
  if constexpr (WAVES == 1) {
    const float top = fmaxf(m, sink);
    const float weight = expf(m - top);
    const float inv = weight / (l * weight + expf(sink - top));
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d < D) o[d] = from_float<T>(acc[i] * inv);
    }
  } else {
    if (lane == 0) {
      m_s[wave] = m;
      l_s[wave] = l;
    }
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d < D) acc_s[wave][d] = acc[i];
    }
    __syncthreads();
    if (wave != 0) return;
    float top = sink;
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, m_s[w]);
    float total = sink == -INFINITY ? 0.f : expf(sink - top);
    float weight[WAVES];
    for (int w = 0; w < WAVES; ++w) {
      weight[w] = m_s[w] == -INFINITY ? 0.f : expf(m_s[w] - top);       // a wave without keys counts nothing
      total += l_s[w] * weight[w];
    }
    const float inv = 1.f / total;
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d >= D) continue;
      float sum = 0.f;
      for (int w = 0; w < WAVES; ++w) sum += acc_s[w][d] * weight[w];
      o[d] = from_float<T>(sum * inv);
    }
  }
}

// The same walk in float32 for requests that decode, with loads that cover whole rows: one workgroup per
// (token, kv head, part of up to G query heads of it). For the scores eight lanes share a key: each reads 16 of every 128 bytes
// of the key's row of K (a load covers whole lines of eight rows) against its columns of the heads' queries, which it keeps in registers;
// the sums of the eight lanes are added by three exchanges. For the output four lanes share a dimension: each reads four of every
// sixteen keys (a load covers 64 bytes of sixteen neighbouring rows of V^T, one run of 1,024 bytes in pages of sixteen tokens), and
// their sums meet when all keys are through. With G > 1 every row of K and every value of V^T is read once for G heads.
//
// What bounds it is the chain of trips to memory that a wave makes for 64 keys (page, K, V) and the lines that its loads touch, so
// the keys of a token can go to gridDim.z workgroups in runs of whole chunks (each token's own keys cut alike), which leave their
// sums for attn_grouped_merge_kernel. `grouped_plan` chooses heads, waves and runs. With a lane on 64 neighbouring bytes of K and on a dimension of V^T
// every load touched 64 lines. us with the merge, K and V from memory, so / now: 12 heads of 128 on 2, 8 requests of 1,000
// keys 13.2 / 10.9, 1 of 500 12.7 / 8.7, 32 of 200 9.6 / 7.3, 32 of 1,000 22.4 / 19.7; 12 of 64, 8 of 1,000 19.7 / 15.4; 8 of 256 on
// 4, 1 of 400 19.0 / 12.7; against 64 bits 2.3e-7 / 2.0e-7.
constexpr bool GQ_FITS = D % 32 == 0;
constexpr int GQ_SLICE = GQ_FITS ? D / 8 : 4;             // a lane's columns of K
constexpr int GQ_DIMS = GQ_FITS ? D / 16 : 1;              // a lane's dimensions of V: lane / 4, 16 more, ...
static bool grouped_fits(int64_t tokens, int heads) { return GQ_FITS && tokens * heads < 2048; }

// (The second bound keeps as many waves a SIMD as there were with fewer sums a lane; for that one register goes to scratch memory with three
// or four query heads of 64 and two or four of 256. With two heads beyond 256 it would be 127 to 489, for one wave a SIMD more.)
template <int G, int WAVES>
__global__ __launch_bounds__(DISTIE_WAVE * WAVES, (D <= 64 ? 4 : G == 2 && D <= 256 ? 2 : 1)) void attn_grouped_f32_kernel(
    const float* __restrict__ qkv, int64_t q_stride, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ token_request,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows,
    float* __restrict__ out, int heads, int kv_heads, int parts, int block_size, float scale, int window,
    const float* __restrict__ sinks, float* __restrict__ part_o, float* __restrict__ part_ml, int runs) {
  __shared__ float p_s[WAVES][G][DISTIE_WAVE];
  __shared__ int64_t base_s[WAVES][DISTIE_WAVE];
  __shared__ float m_s[WAVES][G], l_s[WAVES][G];
  __shared__ float acc_s[WAVES][G][D];
  const int lane = threadIdx.x % DISTIE_WAVE;
  const int wave = threadIdx.x / DISTIE_WAVE;
  const int64_t t = blockIdx.x;
  const int group = heads / kv_heads;
  const int kh = blockIdx.y / parts;
  const int g0 = (blockIdx.y % parts) * G;
  const int n = min(G, group - g0);                        // heads of this part
  const int h0 = kh * group + g0;
  const int q_pos = positions[t];
  const int request_of_token = token_request[t];
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request_of_token] : request_of_token) * table_width;
  const int sub = lane % 8;                                // which 16 bytes of a line
  const int key_in_pass = lane / 8;
  float q_r[G][GQ_SLICE];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float* q = qkv + t * q_stride + static_cast<int64_t>(h0 + min(g, n - 1)) * D + 4 * sub;
#pragma unroll
    for (int d = 0; d < GQ_SLICE; d += 4) {
      const float4 v = *reinterpret_cast<const float4*>(q + 8 * d);
      q_r[g][d] = v.x; q_r[g][d + 1] = v.y; q_r[g][d + 2] = v.z; q_r[g][d + 3] = v.w;
    }
  }
  const int first = first_visible(q_pos, window);
  const int last = q_pos;   // inclusive
  float m[G], l[G];
  float acc[G][GQ_DIMS];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int i = 0; i < GQ_DIMS; ++i) acc[g][i] = 0.f;
  }

  const int chunk0 = first / DISTIE_WAVE, chunks = last / DISTIE_WAVE - chunk0 + 1;
  const int per_run = runs == 1 ? chunks : (chunks + runs - 1) / runs;
  const int run0 = static_cast<int>(blockIdx.z) * per_run;
  const int run_end = min(chunks, run0 + per_run);          // (a run may hold no chunk)
  // What is under way together is what the registers hold without a workgroup less on a compute unit. Heads of up to 128 (and
  // beyond 64, where four waves a SIMD hide more than loads ahead do): all of a chunk's keys and, in their place as they are used up, its
  // values; with three or four query heads half of the keys and of the values at a time.
  constexpr bool AHEAD = D > 64 && D <= 128;
  // Heads beyond 288 don't fit so: their keys go in rounds of at most 72 loads (with two query heads 36, with more 18) and a quarter's
  // values in parts; what does not fit goes through scratch memory. us without / with that: 8 heads of 512 on 4, 8 requests of 1,000 keys
  // 69 / 28, 12 on 4, 32 of 200 98 / 23; 8 of 1,024 on one, 8 of 1,000 340 / 49; 12 of 320 on 4, 8 of 1,000 36.4 / 23.9.
  constexpr int K_ROOM = (G == 1 ? 72 : G <= 2 || D <= 288 ? 36 : 18) / (GQ_SLICE / 4);
  constexpr int ROUND = (G == 1 || (AHEAD && G == 2)) && K_ROOM >= 8 ? 8 : K_ROOM >= 4 ? 4 : K_ROOM >= 2 ? 2 : 1;
  constexpr int V_EARLY = !AHEAD ? 0 : G <= 2 ? 2 : 1;
  constexpr int V_PART = D <= 288 ? GQ_DIMS : G <= 2 ? 16 : 8, V_PARTS = (GQ_DIMS + V_PART - 1) / V_PART;      // dimensions
  constexpr int V_LOADS = G <= (AHEAD ? 2 : 1) ? 16 : 8;       // about, in whole quarters of the chunk
  constexpr int V_QUARTERS = V_LOADS >= 4 * GQ_DIMS ? 4 : V_LOADS >= 2 * GQ_DIMS ? 2 : 1, V_BATCHES = 4 / V_QUARTERS;
  for (int c = (chunk0 + run0 + wave) * DISTIE_WAVE; c < (chunk0 + run_end) * DISTIE_WAVE; c += DISTIE_WAVE * WAVES) {
    // Every load of a phase is issued before its results are used (a chunk costs a few trips to memory, not one
    // for every pass and page): lane j looks up the page of key c + j, the addresses go from lane to lane.
    const int key = c + lane;
    const bool valid = key >= first && key <= last;
    int64_t base = 0, row = 0;                              // keys that do not count read the start of the cache
    if (valid) {
      const int page = table[key / block_size];
      base = (static_cast<int64_t>(page) * kv_heads + kh) * block_size * D;
      row = base + static_cast<int64_t>(key % block_size) * D;
    }
    base_s[wave][lane] = base;
    __builtin_amdgcn_wave_barrier();
    // V^T's loads, sixteen keys a quarter (a lane's four lie in one page: pages hold a multiple of four tokens). No condition
    // stands around a load.
    const int lo = max(first - c, 0);                                   // keys lo .. hi of the chunk count
    const int hi = min(DISTIE_WAVE - 1, last - c);
    const int piece = lane % 4, dim0 = lane / 4;
    float4 vv[4][GQ_DIMS];
    const auto ask_values = [&](int batch, int part) {
#pragma unroll
      for (int u = 0; u < V_QUARTERS; ++u) {
        const int quarter = batch * V_QUARTERS + u, j = 16 * quarter + 4 * piece;
        const int64_t page_base = base_s[wave][min(max(j, lo), hi)];      // of a key that counts
        const float* v = v_cache + page_base + static_cast<int64_t>(dim0) * block_size + (c + j) % block_size;
#pragma unroll
        for (int i = part * V_PART; i < min(GQ_DIMS, (part + 1) * V_PART); ++i)
          vv[quarter][i] = *reinterpret_cast<const float4*>(v + 16 * i * block_size);
      }
    };
    // ---- scores: eight keys a pass, ROUND passes of loads under way together; afterwards lane j holds the scores of key c + j.
    // The first values are asked for behind the last keys, the next ones as each half of those is used up.
    float s[G];
#pragma unroll
    for (int g = 0; g < G; ++g) s[g] = 0.f;
    float4 kk[8][GQ_SLICE / 4];
    const auto ask_keys = [&](int pass) {
      const int64_t from = __shfl(row, 8 * pass + key_in_pass, DISTIE_WAVE);
      const float* k = k_cache + from + 4 * sub;
#pragma unroll
      for (int d = 0; d < GQ_SLICE / 4; ++d) kk[pass][d] = *reinterpret_cast<const float4*>(k + 32 * d);
    };
    const auto use_keys = [&](int pass) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float v = 0.f;
#pragma unroll
        for (int d = 0; d < GQ_SLICE / 4; ++d) {
          v = fmaf(q_r[g][4 * d], kk[pass][d].x, v);
          v = fmaf(q_r[g][4 * d + 1], kk[pass][d].y, v);
          v = fmaf(q_r[g][4 * d + 2], kk[pass][d].z, v);
          v = fmaf(q_r[g][4 * d + 3], kk[pass][d].w, v);
        }
        v = lanes_sum<4>(lanes_sum<2>(lanes_sum<1>(v)));
        if (sub == pass) s[g] = v;                          // lane 8 k + p holds the score of key 8 p + k
      }
    };
#pragma unroll
    for (int round = 0; round < 8 / ROUND; ++round) {
#pragma unroll
      for (int ps = 0; ps < ROUND; ++ps) ask_keys(ROUND * round + ps);
      __builtin_amdgcn_sched_barrier(0);                    // all of these loads are under way before the first is used
#pragma unroll
      for (int ps = 0; ps < ROUND; ++ps) {
        use_keys(ROUND * round + ps);
        if constexpr (V_EARLY > 0) {
          const int half = (ps + 1) / (ROUND / 2) - 1;
          if (round == 8 / ROUND - 1 && (ps + 1) % (ROUND / 2) == 0 && half < V_EARLY) {
            __builtin_amdgcn_sched_barrier(0);
            ask_values(half, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
    float alpha[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      s[g] = __shfl(s[g], sub * 8 + lane / 8, DISTIE_WAVE);
      const float sg = valid && g < n ? s[g] * scale : -INFINITY;
      const float m_new = fmaxf(m[g], wave_max(sg));
      alpha[g] = m_new == -INFINITY ? 0.f : expf(m[g] - m_new);     // 0 on the first chunk with a key (m = -inf)
      const float p = valid && g < n ? expf(sg - m_new) : 0.f;
      l[g] = l[g] * alpha[g] + wave_sum(p);
      m[g] = m_new;
      p_s[wave][g][lane] = p;
    }
    __builtin_amdgcn_wave_barrier();
    // ---- output
#pragma unroll
    for (int batch = 0; batch < V_BATCHES; ++batch) {
#pragma unroll
      for (int part = 0; part < V_PARTS; ++part) {
        if (batch >= V_EARLY) {
          __builtin_amdgcn_sched_barrier(0);
          ask_values(batch, part);
          __builtin_amdgcn_sched_barrier(0);                  // all of these loads are under way before the first is used
        }
        const int first_dim = part * V_PART, end_dim = min(GQ_DIMS, first_dim + V_PART);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (batch == 0) {
#pragma unroll
            for (int i = first_dim; i < end_dim; ++i) acc[g][i] *= alpha[g];
          }
#pragma unroll
          for (int u = 0; u < V_QUARTERS; ++u) {
            const int quarter = batch * V_QUARTERS + u, j = 16 * quarter + 4 * piece;
            const float4 p = *reinterpret_cast<const float4*>(&p_s[wave][g][j]);
            // never a value of a key that does not count (a weight of zero times what lies there could be NaN)
            const bool in[4] = {j >= lo && j <= hi, j + 1 >= lo && j + 1 <= hi, j + 2 >= lo && j + 2 <= hi, j + 3 >= lo && j + 3 <= hi};
#pragma unroll
            for (int i = first_dim; i < end_dim; ++i) {
              const float4 v = vv[quarter][i];
              acc[g][i] = fmaf(p.x, in[0] ? v.x : 0.f, acc[g][i]);
              acc[g][i] = fmaf(p.y, in[1] ? v.y : 0.f, acc[g][i]);
              acc[g][i] = fmaf(p.z, in[2] ? v.z : 0.f, acc[g][i]);
              acc[g][i] = fmaf(p.w, in[3] ? v.w : 0.f, acc[g][i]);
            }
          }
        }
      }
    }
  }
  // ---- the waves' parts, put together by wave 0 in wave order
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m_s[wave][g] = m[g];
      l_s[wave][g] = l[g];
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < GQ_DIMS; ++i) {
      const float sum = lanes_sum<2>(lanes_sum<1>(acc[g][i]));
      if (lane % 4 == 0) acc_s[wave][g][lane / 4 + 16 * i] = sum;
    }
  __syncthreads();
  // wave w writes heads w, w + WAVES, ... of the part
  const bool whole = runs == 1;
  for (int g = wave; g < n; g += WAVES) {
    const float sink = whole && sinks != nullptr ? sinks[h0 + g] : -INFINITY;      // one more term of the denominator, no value
    float top = sink;
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, m_s[w][g]);
    float total = sink == -INFINITY ? 0.f : expf(sink - top);
    float weight[WAVES];
    for (int w = 0; w < WAVES; ++w) {
      weight[w] = m_s[w][g] == -INFINITY ? 0.f : expf(m_s[w][g] - top);    // a wave without keys counts nothing
      total += l_s[w][g] * weight[w];
    }
    const int64_t at = t * heads + h0 + g + (whole ? 0 : static_cast<int64_t>(blockIdx.z) * gridDim.x * heads);
    const float inv = whole ? 1.f / total : 1.f;
    float* o = (whole ? out : part_o) + at * D;
    if (!whole && lane == 0) {
      part_ml[2 * at] = top;
      part_ml[2 * at + 1] = total;
    }
    if (!whole && total == 0.f) continue;                   // no key in this run: its sums are not read
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d >= D) continue;
      float sum = 0.f;
      for (int w = 0; w < WAVES; ++w) sum += acc_s[w][g][d] * weight[w];
      o[d] = sum * inv;
    }
  }
}

// The runs of attn_grouped_f32_kernel put together in their order: a workgroup of one wave a (token, head).
constexpr int GQ_MAX_RUNS = 16;

__global__ __launch_bounds__(DISTIE_WAVE) void attn_grouped_merge_kernel(const float* __restrict__ part_o,
                                                                         const float* __restrict__ part_ml,
                                                                         float* __restrict__ out, int heads, int runs,
                                                                         const float* __restrict__ sinks) {
  const int64_t at = static_cast<int64_t>(blockIdx.x) * heads + blockIdx.y;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * heads;
  float2 ml[GQ_MAX_RUNS];
#pragma unroll
  for (int s = 0; s < GQ_MAX_RUNS; ++s)
    ml[s] = s < runs ? *reinterpret_cast<const float2*>(part_ml + 2 * (s * stride + at)) : float2{-INFINITY, 0.f};
  const float sink = sinks != nullptr ? sinks[blockIdx.y] : -INFINITY;
  float top = sink;
#pragma unroll
  for (int s = 0; s < GQ_MAX_RUNS; ++s) top = fmaxf(top, ml[s].x);
  float total = sink == -INFINITY ? 0.f : expf(sink - top);
  float weight[GQ_MAX_RUNS];
#pragma unroll
  for (int s = 0; s < GQ_MAX_RUNS; ++s) {
    weight[s] = ml[s].y > 0.f ? expf(ml[s].x - top) : 0.f;
    total += ml[s].y * weight[s];
  }
  const float inv = 1.f / total;
  for (int d = 4 * threadIdx.x; d < D; d += 4 * DISTIE_WAVE) {
    float4 o[GQ_MAX_RUNS];
#pragma unroll
    for (int s = 0; s < GQ_MAX_RUNS; ++s) {
      o[s] = float4{0.f, 0.f, 0.f, 0.f};
      if (s < runs && ml[s].y > 0.f) o[s] = *reinterpret_cast<const float4*>(part_o + (s * stride + at) * D + d);
    }
    float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < GQ_MAX_RUNS; ++s) {
      sum.x = fmaf(weight[s], o[s].x, sum.x);
      sum.y = fmaf(weight[s], o[s].y, sum.y);
      sum.z = fmaf(weight[s], o[s].z, sum.z);
      sum.w = fmaf(weight[s], o[s].w, sum.w);
    }
    *reinterpret_cast<float4*>(out + at * D + d) = float4{sum.x * inv, sum.y * inv, sum.z * inv, sum.w * inv};
  }
}

// The same attention on the float32 matrix instruction (v_mfma_f32_16x16x4_f32), for any step: the 16 columns of a
// product are the query heads of one kv head (at most 16 of them) for as many consecutive tokens of a request as fit, so a
// row of K and of V^T is read once for all of them. A workgroup of four waves a (tile of tokens, kv head, run of keys): the
// waves take chunks of CF_KEYS keys in turn, straight from the cache to registers (a lane's 16 bytes are its operand of four
// products: of K's row `lane % 16`, of V^T's row of a dim `lane % 16`), K and V of a chunk asked for together. Scores are
// summed over the head's dimensions in sixteen chains, values
// in one for every 16 keys: no further from 64 bits than the vector kernels. The waves' results are put together in LDS, the runs' by
// attn_grouped_merge_kernel.
constexpr bool CF_FITS = D % 32 == 0 && D <= 256;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float cf_floatx4;
constexpr int CF_WAVES = 4;
constexpr int CF_BLOCKS = D <= 128 ? 4 : 2;               // of 16 keys a chunk: what the registers of one wave a SIMD hold
constexpr int CF_KEYS = 16 * CF_BLOCKS;

__global__ __launch_bounds__(DISTIE_WAVE * CF_WAVES, 1) void attn_columns_f32_kernel(
    const float* __restrict__ qkv, int64_t q_stride, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ block_table,
    int table_width, const int32_t* __restrict__ table_rows, float* __restrict__ out, int tokens, int num_requests, int heads,
    int kv_heads, int block_size, float scale, int window, const float* __restrict__ sinks, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
  if constexpr (CF_FITS) {
  constexpr int DJ = D / 16;
  __shared__ __attribute__((aligned(16))) float acc_s[CF_WAVES][16][D];
  __shared__ float m_s[CF_WAVES][16], l_s[CF_WAVES][16];
  const int lane = threadIdx.x % DISTIE_WAVE;
  const int wave = threadIdx.x / DISTIE_WAVE;
  const int r = lane % 16, g = lane / 16;
  const int kh = blockIdx.y;
  const int group = heads / kv_heads;
  const int most = 16 / group;                              // tokens of a tile
  // ---- which request's tile this is: 64 requests at a time
  int request = -1, tile = blockIdx.x;
  for (int i0 = 0; i0 < num_requests && request < 0; i0 += DISTIE_WAVE) {
    const int i = i0 + lane;
    const int own = i < num_requests ? (cu_q[i + 1] - cu_q[i] + most - 1) / most : 0;
    int upto = own;
#pragma unroll
    for (int o = 1; o < DISTIE_WAVE; o *= 2) {
      const int before = __shfl_up(upto, o, DISTIE_WAVE);
      if (lane >= o) upto += before;
    }
    const uint64_t holds = __ballot(upto > tile);
    if (holds != 0) {
      const int at = __ffsll(static_cast<unsigned long long>(holds)) - 1;
      request = i0 + at;
      tile -= __shfl(upto - own, at, DISTIE_WAVE);
    } else {
      tile -= __shfl(upto, DISTIE_WAVE - 1, DISTIE_WAVE);
    }
  }
  if (request < 0) return;                                  // (the grid is an upper bound)
  const int token0 = cu_q[request] + tile * most;
  const int count = min(most, cu_q[request + 1] - token0);
  const int pos0 = positions[token0];
  const int first = first_visible(pos0, window);
  const int last = pos0 + count - 1;                        // inclusive, of the tile's last token
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request] : request) * table_width;

  // ---- the lane's column: head kh * group + r % group of token token0 + r / group (columns past the end repeat the last)
  const int col = min(r, count * group - 1);
  const int col_last = pos0 + col / group;
  const int col_first = first_visible(col_last, window);
  cf_floatx4 q_reg[DJ];
  {
    const float* q = qkv + (token0 + col / group) * q_stride + static_cast<int64_t>(kh * group + col % group) * D + 4 * g;
#pragma unroll
    for (int j = 0; j < DJ; ++j) q_reg[j] = *reinterpret_cast<const cf_floatx4*>(q + 16 * j);
  }
  const int chunk0 = first / CF_KEYS, chunks = last / CF_KEYS - chunk0 + 1;
  const int per_run = (chunks + static_cast<int>(gridDim.z) - 1) / static_cast<int>(gridDim.z);
  const int run0 = static_cast<int>(blockIdx.z) * per_run;
  const int run_end = min(chunks, run0 + per_run);          // (a run may hold no chunk)
  // All tokens of the tile at once (turn 0). A key that some of them see and some do not weighs zero for those, and zero
  // times a value that is not finite is NaN: a wave whose sums are not all finite takes the tokens again one by one (token
  // turn - 1), each over the keys that it sees. (Only the sums are looked at: a look at V itself would hold more registers
  // than there are at heads of 256. 8 heads of 256 on 1, 5 single tokens and a prompt of 200: 35.1 -> 37.3 us.)
  for (int turn = 0;; ++turn) {
  const int turn_first = turn > 0 ? first_visible(pos0 + turn - 1, window) : first;
  const int turn_last = turn > 0 ? pos0 + turn - 1 : last;
  cf_floatx4 o_acc[DJ];
#pragma unroll
  for (int j = 0; j < DJ; ++j) o_acc[j] = cf_floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;                     // (each lane of a column keeps a part of the sum)
  const int end = min((chunk0 + run_end) * CF_KEYS, turn_last + 1);
  int c = (chunk0 + run0 + wave) * CF_KEYS;
  while (c + CF_KEYS <= turn_first) c += CF_KEYS * CF_WAVES;      // (every chunk of the walk holds a key that counts)
  for (; c < end; c += CF_KEYS * CF_WAVES) {
    // lane j looks up the page of key c + j; keys that do not count read the start of the cache
    const int lo = max(turn_first - c, 0), hi = min(CF_KEYS - 1, turn_last - c);      // keys lo .. hi of the chunk count
    int64_t base = 0;
    if (lane >= lo && lane <= hi)
      base = (static_cast<int64_t>(table[(c + lane) / block_size]) * kv_heads + kh) * block_size * D;
    cf_floatx4 k_reg[CF_BLOCKS][DJ], v_reg[CF_BLOCKS][DJ];
#pragma unroll
    for (int b = 0; b < CF_BLOCKS; ++b) {
      const int key = 16 * b + r;
      const bool counts = key >= lo && key <= hi;
      const int64_t page = __shfl(base, key, DISTIE_WAVE);
      const float* k = k_cache + page + (counts ? (c + key) % block_size : 0) * D + 4 * g;
#pragma unroll
      for (int j = 0; j < DJ; ++j) k_reg[b][j] = *reinterpret_cast<const cf_floatx4*>(k + 16 * j);
    }
#pragma unroll
    for (int b = 0; b < CF_BLOCKS; ++b) {
      // four keys of a dim lie in one page; the page is that of one of them that counts
      const int key = 16 * b + 4 * g;
      const int64_t page = __shfl(base, min(max(key, lo), hi), DISTIE_WAVE);
      const float* v = v_cache + page + static_cast<int64_t>(r) * block_size + (c + key) % block_size;
#pragma unroll
      for (int j = 0; j < DJ; ++j) v_reg[b][j] = *reinterpret_cast<const cf_floatx4*>(v + static_cast<int64_t>(16 * j) * block_size);
    }
    __builtin_amdgcn_sched_barrier(0);                      // all of these loads are under way before the first is used
    // ---- scores: the lane holds keys 16 b + 4 g + i of its column
    cf_floatx4 s[CF_BLOCKS];
    float best = -INFINITY;
#pragma unroll
    for (int b = 0; b < CF_BLOCKS; ++b) {
      cf_floatx4 chain[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) chain[e] = cf_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          chain[4 * (j % 4) + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_reg[b][j][e], q_reg[j][e], chain[4 * (j % 4) + e], 0, 0, 0);
#pragma unroll
      for (int half = 8; half > 1; half /= 2)
#pragma unroll
        for (int e = 0; e < half; ++e) chain[e] += chain[e + half];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = c + 16 * b + 4 * g + i;
        const float v = (chain[0][i] + chain[1][i]) * scale;
        s[b][i] = key >= col_first && key <= col_last ? v : -INFINITY;
        best = fmaxf(best, s[b][i]);
      }
    }
    best = lanes_max<16>(best);
    best = lanes_max<32>(best);
    const float m_new = fmaxf(m_run, best);
    const float alpha = m_new == -INFINITY ? 0.f : expf(m_run - m_new);      // 0 on the first chunk with a key (m = -inf)
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < CF_BLOCKS; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = c + 16 * b + 4 * g + i;
        s[b][i] = key >= col_first && key <= col_last ? expf(s[b][i] - m_new) : 0.f;
        sum += s[b][i];
      }
    l_run = l_run * alpha + sum;
    m_run = m_new;
    float a4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a4[i] = __shfl(alpha, 4 * g + i, DISTIE_WAVE);
    // ---- O += P . V: the lane ends with columns 4 g + i of dim 16 j + r; a sum of its own for every 16 keys, added in pairs
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      cf_floatx4 part[CF_BLOCKS];
#pragma unroll
      for (int b = 0; b < CF_BLOCKS; ++b) {
        part[b] = cf_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = 16 * b + 4 * g + i;
          // never a value of a key that does not count (a weight of zero times what lies there could be NaN)
          const float v = key >= lo && key <= hi ? v_reg[b][j][i] : 0.f;
          part[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[b][i], v, part[b], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sum4 = part[0][i] + part[1][i];
        if constexpr (CF_BLOCKS == 4) sum4 += part[2][i] + part[3][i];
        o_acc[j][i] = fmaf(o_acc[j][i], a4[i], sum4);
      }
    }
  }
  l_run = lanes_sum<16>(l_run);
  l_run = lanes_sum<32>(l_run);
  // columns first_col .. end_col are this turn's
  const int first_col = turn > 0 ? (turn - 1) * group : 0, end_col = turn > 0 ? turn * group : 16;
  if (g == 0 && r >= first_col && r < end_col) {
    m_s[wave][r] = m_run;
    l_s[wave][r] = l_run;
  }
  float zero = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < DJ; ++j) zero = fmaf(o_acc[j][i], 0.f, zero);
    if (4 * g + i < first_col || 4 * g + i >= end_col) continue;
#pragma unroll
    for (int j = 0; j < DJ; ++j) acc_s[wave][4 * g + i][16 * j + r] = o_acc[j][i];
  }
  if (turn == 0 ? count == 1 || __all(zero == 0.f) : turn == count) break;
  }
  __syncthreads();
  // ---- the waves' parts, in wave order; four dims of a column a thread
  const bool whole = gridDim.z == 1;
  for (int idx = threadIdx.x; idx < count * group * (D / 4); idx += DISTIE_WAVE * CF_WAVES) {
    const int cl = idx / (D / 4), d = 4 * (idx % (D / 4));
    const int head = kh * group + cl % group;
    const float sink = whole && sinks != nullptr ? sinks[head] : -INFINITY;      // one more term of the denominator, no value
    float top = sink;
#pragma unroll
    for (int w = 0; w < CF_WAVES; ++w) top = fmaxf(top, m_s[w][cl]);
    float total = sink == -INFINITY ? 0.f : expf(sink - top);
    float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < CF_WAVES; ++w) {
      const float weight = m_s[w][cl] == -INFINITY ? 0.f : expf(m_s[w][cl] - top);      // a wave without keys counts nothing
      const float4 o = *reinterpret_cast<const float4*>(&acc_s[w][cl][d]);
      total += l_s[w][cl] * weight;
      sum.x = fmaf(weight, o.x, sum.x);
      sum.y = fmaf(weight, o.y, sum.y);
      sum.z = fmaf(weight, o.z, sum.z);
      sum.w = fmaf(weight, o.w, sum.w);
    }
    const int64_t at = static_cast<int64_t>(token0 + cl / group) * heads + head +
                       (whole ? 0 : static_cast<int64_t>(blockIdx.z) * tokens * heads);
    const float inv = whole ? 1.f / total : 1.f;
    if (!whole && d == 0) {
      part_ml[2 * at] = top;
      part_ml[2 * at + 1] = total;
    }
    *reinterpret_cast<float4*>((whole ? out : part_o) + at * D + d) = float4{sum.x * inv, sum.y * inv, sum.z * inv, sum.w * inv};
  }
  }
}

// Into how many runs distie_attention_columns_f32 is to cut each tile's keys: enough workgroups for every compute unit twice
// over, a round of the four waves each at least; 0 where the step is not for it: few pairs of token and head up to heads of
// 128 (the chain of attn_grouped_f32_kernel is shorter: 8 requests of 1,000 keys, 12 of 128 on 2 14.3 us, would be 19.2), beyond
// 128 single tokens with few heads to share a row (8 on 4, 8 requests: 22.8, would be 24.0), more pairs where a single token
// and a head of its own each fill one column of sixteen (300 requests of 600 keys, 8 on 8: 389, would be 397). Where it may
// be taken, distie_attention_columns_f32_pays says whether it is.
extern "C" int distie_attention_columns_f32_runs(int tokens, int num_requests, int heads, int kv_heads, int block_size,
                                                 int64_t q_stride, int visible) {
  if (!CF_FITS || tokens < 1 || num_requests < 1 || heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || kv_heads > 65535 ||
      heads / kv_heads > 16 || block_size < 4 || block_size % 4 != 0 || q_stride % 4 != 0)
    return 0;
  const int group = heads / kv_heads;
  const bool fills = grouped_fits(tokens, heads) ? D > 128 && (group >= 4 || tokens / 2 >= num_requests)
                                                 : group >= 2 || tokens > num_requests;
  if (!fills) return 0;
  const int64_t tiles = tokens == num_requests ? tokens : tokens / (16 / group) + num_requests;
  const int64_t wanted = (512 + tiles * kv_heads - 1) / (tiles * kv_heads);
  constexpr int ROUND = CF_WAVES * CF_KEYS;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({wanted, (visible + ROUND - 1) / ROUND, GQ_MAX_RUNS})));
}

// Attention of a float32 step whose requests' tokens are rows cu_q[i] .. cu_q[i + 1] at consecutive positions (plain scores,
// a float32 cache). runs > 1: part_o (float32 [runs, tokens, heads, D]) and part_ml (float32 [runs, tokens, heads, 2]).
extern "C" int distie_attention_columns_f32(const void* qkv, int64_t q_stride, const void* k_cache, const void* v_cache,
                                            const int32_t* positions, const int32_t* cu_q, const int32_t* block_table,
                                            int table_width, const int32_t* table_rows, void* out, int tokens, int num_requests,
                                            int heads, int kv_heads, int block_size, float scale, int window, const float* sinks,
                                            float* part_o, float* part_ml, int runs, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (distie_attention_columns_f32_runs(tokens, num_requests, heads, kv_heads, block_size, q_stride, 1) < 1 || table_width < 1 ||
      heads > 65535 || runs < 1 || runs > GQ_MAX_RUNS || (runs > 1 && (part_o == nullptr || part_ml == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const int most = 16 / (heads / kv_heads);
  const int tiles = tokens == num_requests ? tokens : tokens / most + num_requests;      // an upper bound; spare blocks leave at once
  attn_columns_f32_kernel<<<dim3(tiles, kv_heads, runs), DISTIE_WAVE * CF_WAVES, 0, stream>>>(
      static_cast<const float*>(qkv), q_stride, static_cast<const float*>(k_cache), static_cast<const float*>(v_cache), positions,
      cu_q, block_table, table_width, table_rows, static_cast<float*>(out), tokens, num_requests, heads, kv_heads, block_size,
      scale, window, sinks, part_o, part_ml);
  if (runs > 1)
    attn_grouped_merge_kernel<<<dim3(tokens, heads), DISTIE_WAVE, 0, stream>>>(part_o, part_ml, static_cast<float*>(out), heads,
                                                                               runs, sinks);
  return launch_status();
}

// How attn_grouped_f32_kernel takes a step: query heads to a workgroup, its waves, and the runs of keys.
struct GroupedPlan {
  int per, waves, runs;
};

// visible: the most keys that a token sees. From 650 steps (1 to 128 requests of 30 to 16,000 keys, portions of up to 31
// tokens, heads of 64 to 256, groups of 1 to 8; K and V from memory), each with every number of heads, 4 and 8 waves, 1 to 16
// runs; what this takes is 2 % from the best of them on average. us, one run of eight waves a workgroup / this:
//  * runs cost a merge and its launch, some 4.5 us, so keys are cut only where one run has eight waves take two chunks each:
//    1 request, 12 heads of 128 on 2: 200 keys 8.6 / 8.4, 400 keys 11.9 / 11.9 (two runs: 14.2), 700 keys 16.0 / 11.8, 1,000 keys
//    24.9 / 13.9, 4,000 keys 82 / 15.2. Runs of one chunk a wave, or of as many as the chip has room for: 512 workgroups of
//    four waves, fewer where contexts are short for heads of 64 or the registers hold one wave a SIMD, more for long ones;
//    Heads of 96 and 128 then take as many runs as there is room for: a captured step is made for longer contexts than it
//    holds, and of 100 steps of 300 to 5,400 keys (half of them under twice the bound) none was more than 1 % slower, the
//    rest by up to 28 % faster (24 requests of 1,050 keys planned for 2,048, 16 heads on 4: 29 -> 22 us). Heads of 64 do not:
//    up to 16 % slower where the bound is the context (17 requests of 4,600 keys, 16 on 4: 33, would be 38);
//  * heads share a workgroup, and a row of K its load, as far as the chip is full without it: 64 requests of 128 keys, 12 heads
//    of 128 on 2 14.9 / 11.8; a head to itself otherwise (8 requests of 128 keys 8.8 / 8.6, in threes 11.2);
//  * without runs four waves for up to four chunks, then eight, but for more workgroups than compute units, which run two at a
//    time (64 requests of 700 keys, 28 heads of 128 on 4: 57 / 47), and where eight waves do not fit the registers: beyond 128
//    (runs from five chunks on there: 8 heads of 256 on 4, 1 request of 400 keys 38 / 21), and at 96, where the compiler then
//    spills, with more than one head (156 requests of 500 keys, 8 of 96 on 2: 112 / 48).
constexpr int GQ_EIGHT_HEADS = D > 128 ? 0 : D <= 64 || D == 128 ? 4 : 1;      // heads with which eight waves fit
static GroupedPlan grouped_plan(int64_t tokens, int heads, int kv_heads, int visible) {
  const int group = heads / kv_heads, most = std::min(4, group), chunks = (visible + DISTIE_WAVE - 1) / DISTIE_WAVE;
  const int64_t pairs = tokens * kv_heads;
  const auto parts = [&](int per) { return (group + per - 1) / per; };
  const auto even = [&](int per) { return (group + parts(per) - 1) / parts(per); };      // as many heads in each part
  const auto fewest = [&](int64_t limit, int runs) {          // heads a workgroup with which there are at most `limit`; 0: none
    for (int per = 1; per <= most; ++per)
      if (pairs * parts(per) * runs <= limit) return per;
    return 0;
  };
  constexpr bool WIDE = D > 128, NARROW = D <= 64;
  if (chunks > (WIDE ? 4 : most == 1 ? 6 : 8)) {
    const bool lasting = chunks > 18;
    const int64_t apart = NARROW && lasting ? 512 : 256;              // workgroups up to which heads are kept apart
    const int64_t room = NARROW ? (!lasting ? 256 : most == 4 ? 1024 : 512) : D > 192 && !lasting ? 320 : 512;
    const auto filled = [&](int per, int64_t limit, int runs) {          // as many as there is room for, a chunk a wave or more
      if (NARROW || WIDE) return runs;
      return std::max(runs, static_cast<int>(std::min<int64_t>({GQ_MAX_RUNS, limit / (pairs * parts(per)), chunks / 4})));
    };
    for (int trips = 1;; ++trips) {                             // chunks that a wave takes one after the other
      const int runs = std::min(GQ_MAX_RUNS, (chunks + 4 * trips - 1) / (4 * trips));
      // two runs of four waves are one run of eight, where those fit; side by side they spread better for heads of their own
      const bool two = WIDE || (most == 1 && trips == 1);
      if (runs < (two ? 2 : 3)) break;
      const int per = fewest(apart, runs);
      if (per > 0) return {even(per), 4, filled(per, parts(per) == parts(most) ? room : apart, runs)};
      if (pairs * parts(most) * runs <= room && (WIDE || runs > 2)) return {even(most), 4, filled(most, room, runs)};
    }
  }
  const bool four = WIDE || chunks <= 4;
  int per = fewest(NARROW && four ? 512 : 256, 1);
  // more workgroups than compute units: those of eight waves run one at a time at heads of 128, two at 64
  const bool crowded = per == 0 && !(NARROW && pairs * parts(most) <= 512) && most > 1;
  if (per == 0) per = most;
  return {even(per), four || crowded || even(per) > GQ_EIGHT_HEADS ? 4 : 8, 1};
}

// Whether distie_attention_columns_f32 in so many runs is faster than the kernels that take the step otherwise, by what each
// is reckoned to take: whole rounds of workgroups on the compute units (the last one counted half empty), each as long as its
// waves' trips to memory for a chunk of keys, and the merge of runs. A least-squares fit to 700 steps timed both ways (1 to 400
// requests of 8 to 2,500 keys, portions of up to 30 tokens, heads of 32 to 256, groups of 1 to 16), off by 11 to 20 %; with a
// tenth of doubt against the columns what it chooses takes 1 % more than the faster of the two on average. us, columns / otherwise:
//  * short contexts, where a chunk of columns is mostly empty, stay: 8 heads of 256 on 1, 1 request of 24 keys 12.0 / 9.9; 24 on 2
//    of 192, 6 of 139 15.9 / 8.8; 16 on 8 of 64, 259 requests of 13 keys 74 / 10; 28 on 4 of 128, 82 of 21 24 / 12;
//  * many tokens with longer ones, and wide heads, go: 28 on 4 of 64, 151 requests of 1,000 keys 87 / 340; 8 on 1 of 256, 79 of
//    2,000 92 / 136; 12 on 2 of 256, portions of up to 44 tokens behind 300 keys 91 / 432.
// visible: the most keys that a token sees, or, behind a window, that its chunks hold.
extern "C" int distie_attention_columns_f32_pays(int tokens, int num_requests, int heads, int kv_heads, int block_size, int visible,
                                                 int runs) {
  if (tokens < 1 || num_requests < 1 || heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || heads / kv_heads > 16 || visible < 1 ||
      runs < 1)
    return 0;
  const bool few = grouped_fits(tokens, heads);
  if (few && (block_size < 1 || DISTIE_WAVE % block_size != 0)) return 1;       // (attn_grouped_f32_kernel does not take it)
  const int group = heads / kv_heads;
  const int64_t pairs = static_cast<int64_t>(tokens) * heads;
  const auto rounds = [](int64_t workgroups) {
    const float x = static_cast<float>(workgroups) / 256;
    return std::max(1.f, 0.5f * (x + static_cast<float>((workgroups + 255) / 256)));
  };
  const auto trips = [&](int chunk, int cut, int waves) {
    const int chunks = (visible + chunk - 1) / chunk, of_run = (chunks + cut - 1) / cut;
    return static_cast<float>((of_run + waves - 1) / waves);
  };
  const auto merge = [&](float start, float each, int cut) { return cut > 1 ? start + each * pairs * cut * D * 1e-6f : 0.f; };
  constexpr float WIDTH = D / 256.f;
  const int64_t tiles = tokens == num_requests ? tokens : tokens / (16 / group) + num_requests;
  float columns, otherwise;
  if (few) {
    const GroupedPlan plan = grouped_plan(tokens, heads, kv_heads, visible);
    const int64_t workgroups = static_cast<int64_t>(tokens) * kv_heads * ((group + plan.per - 1) / plan.per) * plan.runs;
    otherwise = -2.3f + rounds(workgroups) * (4.05f + trips(DISTIE_WAVE, plan.runs, plan.waves) * (5.75f + 3.75f * plan.per)) * WIDTH +
                merge(5.6f, 11.5f, plan.runs);
    columns = 3.3f + rounds(tiles * kv_heads * runs) * 10.5f * trips(CF_KEYS, runs, CF_WAVES) * WIDTH;
  } else {
    // a wave a pair, sixteen of them on a compute unit, key after key
    const float start = D <= 64 ? 2.35f : D <= 128 ? 1.35f : 2.5f, key0 = D <= 128 ? 6.65f : 8.35f;
    otherwise = start + std::max(1.f, static_cast<float>(pairs) / 4096) * (key0 + 1.05f * visible) * WIDTH;
    columns = (D <= 64 ? 3.9f : D <= 128 ? 6.1f : 8.9f) + rounds(tiles * kv_heads * runs) *
              (D <= 64 ? 27.7f : D <= 128 ? 22.f : 10.1f) * trips(CF_KEYS, runs, CF_WAVES) * WIDTH;
  }
  return columns + merge(5.f, 7.3f, runs) < 0.92f * otherwise;
}

// The plan for a step of distie_attention_generic (float32, plain scores): -> runs, which the caller has buffers for; what a plan
// changes in the results is their rounding. 1 and no heads where another kernel takes the step.
extern "C" int distie_attention_f32_plan(int tokens, int heads, int kv_heads, int visible, int* per, int* waves) {
  *per = *waves = 0;
  if (tokens < 1 || heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || visible < 1 || !grouped_fits(tokens, heads)) return 1;
  const GroupedPlan plan = grouped_plan(tokens, heads, kv_heads, visible);
  *per = plan.per, *waves = plan.waves;
  return plan.runs;
}

// qkv: [T, q_stride] with q of head h at columns h*D; out: [T, heads*D]. window: see the head of the file.
// head_slopes (float32 [heads], may be null): score += slope[h] * (key - position); score_cap > 0: the scaled score
// goes through cap * tanh(score / cap) first. Only this kernel takes the two. sinks (float32 [heads], may be null): the
// softmax's denominator holds exp(sinks[h]) beside the keys' terms; every kernel of this file takes them.
// runs, per, waves: of distie_attention_f32_plan (1, 0, 0: none); runs > 1: part_o (float32 [runs, T, heads, D]) and part_ml
// (float32 [runs, T, heads, 2]).
extern "C" int distie_attention_generic(const void* qkv, int dtype, int64_t q_stride, const void* k_cache,
                                        const void* v_cache, int cache_dtype, const int32_t* positions,
                                        const int32_t* token_request, const int32_t* block_table,
                                        int table_width, const int32_t* table_rows, void* out, int tokens, int heads, int kv_heads,
                                        int block_size, float scale, int window, const float* head_slopes,
                                        float score_cap, const float* sinks, float* part_o, float* part_ml, int runs, int per,
                                        int waves, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || block_size < 1 || table_width < 1 ||
      score_cap < 0.f || runs < 1 || runs > GQ_MAX_RUNS || (runs > 1 && (part_o == nullptr || part_ml == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const bool plain_scores = head_slopes == nullptr && score_cap == 0.f;
  if (heads > 65535) return DISTIE_BAD_ARGUMENT;
  dim3 grid(tokens, heads);
  const int group = heads / kv_heads;
  if (plain_scores && grouped_fits(tokens, heads) && dtype == DISTIE_F32 && cache_dtype == DISTIE_F32 && q_stride % 4 == 0 &&
      block_size % 4 == 0 && DISTIE_WAVE % block_size == 0 && per != 0) {
    // few pairs of token and head, as when requests decode, float32
    if (per < 1 || per > std::min(4, group) || (waves != 4 && (waves != 8 || per > GQ_EIGHT_HEADS))) return DISTIE_BAD_ARGUMENT;
    const int parts = (group + per - 1) / per;
    const dim3 grouped(tokens, kv_heads * parts, runs);
#define DISTIE_GROUPED(G, WAVES)                                                                                   \
    attn_grouped_f32_kernel<G, WAVES><<<grouped, DISTIE_WAVE * WAVES, 0, stream>>>(                                 \
        static_cast<const float*>(qkv), q_stride, static_cast<const float*>(k_cache),                               \
        static_cast<const float*>(v_cache), positions, token_request, block_table, table_width, table_rows,         \
        static_cast<float*>(out), heads, kv_heads, parts, block_size, scale, window, sinks, part_o, part_ml, runs)
#define DISTIE_GROUPED_OF(WAVES, MOST)                                                                             \
    if (per == 1) DISTIE_GROUPED(1, WAVES);                                                                         \
    if constexpr (MOST > 1) {                                                                                      \
      if (per == 2) DISTIE_GROUPED(2, WAVES);                                                                       \
      if (per == 3) DISTIE_GROUPED(3, WAVES);                                                                       \
      if (per == 4) DISTIE_GROUPED(4, WAVES);                                                                       \
    }
    if (waves == 4) {
      DISTIE_GROUPED_OF(4, 4);
    } else if constexpr (GQ_EIGHT_HEADS > 0) {
      DISTIE_GROUPED_OF(8, GQ_EIGHT_HEADS);
    }
#undef DISTIE_GROUPED_OF
#undef DISTIE_GROUPED
    if (runs > 1)
      attn_grouped_merge_kernel<<<dim3(tokens, heads), DISTIE_WAVE, 0, stream>>>(part_o, part_ml, static_cast<float*>(out),
                                                                                 heads, runs, sinks);
    return launch_status();
  }
  // few (token, head) pairs, as when requests decode: eight waves share each pair's keys
  if (static_cast<int64_t>(tokens) * heads < 2048) {
    DISTIE_DISPATCH(dtype, T, DISTIE_DISPATCH(cache_dtype, C,
        (attn_generic_kernel<T, C, 8><<<grid, DISTIE_WAVE * 8, 0, stream>>>(
            static_cast<const T*>(qkv), q_stride, static_cast<const C*>(k_cache), static_cast<const C*>(v_cache),
            positions, token_request, block_table, table_width, table_rows, static_cast<T*>(out), heads, kv_heads, block_size,
            scale, window, head_slopes, score_cap, sinks))));
  } else {
    DISTIE_DISPATCH(dtype, T, DISTIE_DISPATCH(cache_dtype, C,
        (attn_generic_kernel<T, C, 1><<<grid, DISTIE_WAVE, 0, stream>>>(
            static_cast<const T*>(qkv), q_stride, static_cast<const C*>(k_cache), static_cast<const C*>(v_cache),
            positions, token_request, block_table, table_width, table_rows, static_cast<T*>(out), heads, kv_heads, block_size,
            scale, window, head_slopes, score_cap, sinks))));
  }
  return launch_status();
}

#if DISTIE_MATRIX_CORE_ATTENTION
// ===================================================================================================
//  Matrix-core kernels (bfloat16, pages of a multiple of 16 tokens). The decode kernel works on 16-wide
//  blocks of "columns" against blocks of 16 keys with two products (the tiled kernel for portions of prompts
//  does the same with 32-wide blocks and is described where it stands):
//        S^T[key, col] = K[key, :] . q[col, :]        (v_mfma_f32_16x16x32_bf16, K rows as the A operand)
//        online softmax over keys, per column, in float32 (weights as 2^x: scores are scaled by log2 e)
//        O[col, d]  += P[col, key] . V^T[d, key]      (values are stored transposed inside a page, so the
//                                                      summed index, the key, is contiguous for the B operand)
//  A lane holds, of a 16 x 16 score tile, keys 4g..4g+3 of column r (r = lane % 16, g = lane / 16): exactly
//  the shape of the A operand of the second product if its 32 summed keys are taken in the order
//  (block 0: 4g..4g+3, block 1: 4g..4g+3); the values are read in the same order, so no data moves
//  between lanes except the maxima and the rescaling factors.
//
//  * attn_decode: requests that bring one token. Columns = the G query heads that share one kv head. The
//    keys of a request are cut into runs of equal length, one wave each (this is where the parallelism comes from when
//    few requests decode); a wave takes its run in chunks of DC_KEYS keys and issues every load of a chunk
//    (pages, K rows, V^T rows) before it computes, so a chunk costs one trip to memory. It writes
//    unnormalised partial results that attn_reduce combines.
// ===================================================================================================
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short shortx4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t uintx4;

// 2^x in one instruction (v_exp_f32; float32, about 1 ulp; -inf gives 0)
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int DK32 = D / 32;            // full 32-wide steps of the q.k product
constexpr bool DK_TAIL = (D % 32) != 0; // one more step of 16
constexpr int DB16 = D / 16;            // 16-wide blocks of the output
constexpr int DC_BLOCKS = (D <= 128) ? 4 : 2;   // blocks of 16 keys whose loads are in flight together
constexpr int DC_KEYS = 16 * DC_BLOCKS;

// What a sink does to a finished column: with the keys' maximum m and sum l (in units of log 2, l relative to m) and the
// sink z (the same units; -inf: none), the factor on the unnormalised output is 2^(m - top) / (l 2^(m - top) + 2^(z - top)),
// top = max(m, z): exp(z) is one more term of the denominator and has no value.
__device__ __forceinline__ float sink_factor(float m, float l, float sink2) {
  if (sink2 == -INFINITY) return 1.f / l;
  const float top = fmaxf(m, sink2);
  const float weight = m == -INFINITY ? 0.f : fast_exp2(m - top);
  return weight / (l * weight + fast_exp2(sink2 - top));
}

// How one request's keys are cut into runs. The visible keys (all of them, or the window's), counted from the
// 64-key boundary at or before the first of them, are cut into at most `max_splits` runs of one length, a
// multiple of RUN_STEP: the request's own length decides, not the longest of the batch, so that every request
// keeps all of its waves busy whatever else the step holds. Both kernels derive the same numbers.
constexpr int RUN_STEP = 64;            // a multiple of DC_KEYS for every head size
struct KeyRuns {
  int first;      // first visible key
  int origin;     // where run 0 begins
  int length;     // keys per run
  int count;      // runs that hold a key
};
// run_len > 0: runs of this length for every request (`decode_run_len_kernel`), so that a long request gets more of them
// than a short one; the caller made it long enough for the longest request to fit max_splits runs.
__device__ __forceinline__ KeyRuns key_runs(int q_pos, int window, int max_splits, int run_len = 0) {
  KeyRuns runs;
  runs.first = first_visible(q_pos, window);
  runs.origin = runs.first / RUN_STEP * RUN_STEP;
  const int span = q_pos - runs.origin + 1;
  const int step = max_splits * RUN_STEP;
  runs.length = run_len > 0 ? run_len : (span + step - 1) / step * RUN_STEP;        // ceil(span / max_splits), rounded up to RUN_STEP
  runs.count = (span + runs.length - 1) / runs.length;      // <= max_splits
  return runs;
}

// One run length for all requests of a step (no window): the shortest, in steps of 64 keys, with which the runs of
// all requests together are at most `budget` (the waves the caller wants at work, per kv head) and no request has
// more than `max_splits`. A long request then gets more runs than a short one; with every request cut into the
// same number of runs the runs of the longest end last, alone. The caller uses it where that same number would
// leave many of the waves unused (256 requests of 1,050 to 3,150 keys on 4 kv heads, one run each: 263 us, with one
// run length 245); requests of one length are cut exactly as without it. It is the same for every layer of a step,
// so one wave finds it once a step and the attention kernels read it beside their request's length (found by
// every wave of theirs it cost 3 to 10 us a call).
__global__ __launch_bounds__(DISTIE_WAVE) void decode_run_len_kernel(const int32_t* __restrict__ kv_len, int num_requests,
                                                                     int budget, int max_splits, int32_t* __restrict__ run_len) {
  const int lane = threadIdx.x;
  int most = 1;
  for (int i = lane; i < num_requests; i += DISTIE_WAVE) most = max(most, kv_len[i]);
#pragma unroll
  for (int o = DISTIE_WAVE / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, DISTIE_WAVE));
  // in units of RUN_STEP keys: from what the longest request needs to fit max_splits runs, up to one run a request
  int lo = (most + max_splits * RUN_STEP - 1) / (max_splits * RUN_STEP);
  int hi = (most + RUN_STEP - 1) / RUN_STEP;
  while (lo < hi) {                                     // (the same in every lane)
    const int mid = (lo + hi) / 2;
    int runs = 0;
    for (int i = lane; i < num_requests; i += DISTIE_WAVE) runs += (kv_len[i] + mid * RUN_STEP - 1) / (mid * RUN_STEP);
#pragma unroll
    for (int o = DISTIE_WAVE / 2; o > 0; o >>= 1) runs += __shfl_xor(runs, o, DISTIE_WAVE);
    if (runs <= budget) {
      hi = mid;
    } else {
      lo = mid + 1;
    }
  }
  if (lane == 0) *run_len = lo * RUN_STEP;
}

// run_len: int32 [1], for a step of num_requests requests that bring one token each.
extern "C" int distie_attention_decode_run_len(const int32_t* kv_len, int num_requests, int budget, int max_splits,
                                               int32_t* run_len, hipStream_t stream) {
  if (num_requests < 1 || budget < 1 || max_splits < 1 || kv_len == nullptr || run_len == nullptr) return DISTIE_BAD_ARGUMENT;
  decode_run_len_kernel<<<1, DISTIE_WAVE, 0, stream>>>(kv_len, num_requests, budget, max_splits, run_len);
  return launch_status();
}

// What bounds a short run is its trips to memory, so all loads of a chunk go out together (48 at a head size of 128; only then are the
// values behind the run's end cleared, and no load stands under a condition). With each block of 16 keys under a condition of its own
// and its values cleared as they came, the compiler waited for every block before it asked for the next, and for every one of the last
// 16 values of a head of 256: us a layer in a step, before / now:
// 16 heads of 256 on one, 16 requests of 1,500 keys 23.2 / 10.0; 12 heads of 128 on 2, one request of 500 keys 6.5 / 4.8, 8 of 2,048
// 7.9 / 6.7, 64 of 2,048 28.2 / 28.2 (that is 4.8 TB/s).
// Two waves a SIMD where the registers allow it without spilling (one block of query heads, head sizes up to 128:
// 206 registers). The chip then holds 2,048 waves
// instead of 1,024, and a batch whose runs are a few more than 1,024, or whose requests differ in length, no
// longer waits for the last waves to get a place: 7B shape's heads at 2,100 keys, 96 requests 91 -> 83 us a layer,
// 160 requests 165 -> 130; contexts of 1,050 to 3,150 keys, 96 requests 121 -> 96, 160 requests 222 -> 157.
template <int MB, int W>
__global__ __launch_bounds__(DISTIE_WAVE * W, (MB == 1 && D <= 128 ? 2 : 1)) void attn_decode_kernel(
    const bf16_t* __restrict__ qkv, int64_t q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ kv_len, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows, float* __restrict__ part_o,
    float* __restrict__ part_ml, int heads, int kv_heads, int block_size, float scale, int window, int split_hint,
    int max_splits, int dense_rows, const int32_t* __restrict__ shared_run_len) {
  const int lane = W > 1 ? threadIdx.x % DISTIE_WAVE : threadIdx.x;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / DISTIE_WAVE) : 0;
  const int r = lane % 16;
  const int g = lane / 16;
  const int group = heads / kv_heads;
  const float scale_log2 = scale * 1.4426950408889634f;
  // With a shared run length the run is the slowest index of the grid: the places past a request's last run, whose
  // waves leave at once, then come after all the others (in front of them they held the places on the SIMDs that
  // the working waves behind them were waiting for: 64 requests took 106 us instead of 54, at one wave a SIMD).
  const bool shared = shared_run_len != nullptr;
  const int share = shared ? blockIdx.z : blockIdx.x;        // the runs W share .. W share + W - 1, one a wave
  const int run = W * share + wave;
  const int request = shared ? blockIdx.y : blockIdx.z;
  const int kh = shared ? blockIdx.x : blockIdx.y;
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request] : request) * table_width;
  // The pages of the run's first chunk are asked for before the request's length says where the run begins:
  // at the place it has if the runs are `split_hint` long and begin at key 0, which the host derives from the
  // longest request of the step (the entry is inside the table either way). Where the guess holds, which it
  // does when few requests of similar length decode, that is one trip to memory less on the way to the keys.
  const int guess_begin = run * split_hint;
  int pages[DC_BLOCKS];
#pragma unroll
  for (int b = 0; b < DC_BLOCKS; ++b) pages[b] = table[min((guess_begin + 16 * b) / block_size, table_width - 1)];
  // dense_rows: every request brings one token, so request i's token is row i
  const int run_len = shared ? *shared_run_len : 0;
  const int token = dense_rows ? request : cu_q[request];
  if (!dense_rows && cu_q[request + 1] - token != 1) return;        // a portion of a prompt: the tiled kernel's
  const int q_pos = kv_len[request] - 1;              // the new token is the last one cached
  const KeyRuns runs = key_runs(q_pos, window, max_splits, run_len);
  if (W * share >= runs.count) return;
  const int run_begin = runs.origin + run * runs.length;
  const int key_begin = max(runs.first, run_begin);
  // (a wave past the last run has no key)
  const int key_end = W == 1 || run < runs.count ? min(q_pos, run_begin + runs.length - 1) : -1;

  // ---- the query of this lane's column (head kh * G + 16 mb + r; columns past the group repeat the last)
  bf16x8 q_reg[MB][DK32 > 0 ? DK32 : 1];
  shortx4 q_tail[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int col = min(16 * mb + r, group - 1);
    const bf16_t* q = qkv + token * q_stride + static_cast<int64_t>(kh * group + col) * D;
#pragma unroll
    for (int dk = 0; dk < DK32; ++dk) q_reg[mb][dk] = *reinterpret_cast<const bf16x8*>(q + 32 * dk + 8 * g);
    if (DK_TAIL) q_tail[mb] = *reinterpret_cast<const shortx4*>(q + (D - 16) + 4 * g);
  }
  floatx4 o_acc[MB][DB16];
  float m_run[MB], l_run[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    m_run[mb] = -INFINITY;
    l_run[mb] = 0.f;
#pragma unroll
    for (int db = 0; db < DB16; ++db) o_acc[mb][db] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // every chunk of the walk holds at least one visible key (the running maximum is then finite): under a
  // window the walk starts at the chunk of the first visible key, whose pages are asked for now
  const int chunk_begin = max(run_begin, key_begin / DC_KEYS * DC_KEYS);      // runs begin at multiples of DC_KEYS
  if (chunk_begin != guess_begin) {
#pragma unroll
    for (int b = 0; b < DC_BLOCKS; ++b) pages[b] = table[min((chunk_begin + 16 * b) / block_size, table_width - 1)];
  }
  for (int chunk = chunk_begin; chunk <= key_end; chunk += DC_KEYS) {
    // ---- every load of the chunk first, none of them under a condition: a block outside the run, which may have no page, reads
    // the nearest one inside again
    const int low = max(key_begin - chunk, 0) / 16, high = min((key_end - chunk) / 16, DC_BLOCKS - 1);
    bf16x8 k_reg[DC_BLOCKS][DK32 > 0 ? DK32 : 1];
    shortx4 k_tail[DC_BLOCKS];
    uint2 v_reg[DC_BLOCKS][DB16];
    const bf16_t* v_from[DC_BLOCKS];
#pragma unroll
    for (int b = 0; b < DC_BLOCKS; ++b) {
      const int inside = min(max(b, low), high);
      int page = pages[0];
#pragma unroll
      for (int i = 1; i < DC_BLOCKS; ++i) page = inside == i ? pages[i] : page;
      const int64_t page_base = (static_cast<int64_t>(page) * kv_heads + kh) * block_size * D;
      const int offset = (chunk + 16 * inside) % block_size;
      const bf16_t* k_row = k_cache + page_base + static_cast<int64_t>(offset) * D;
#pragma unroll
      for (int dk = 0; dk < DK32; ++dk) k_reg[b][dk] = *reinterpret_cast<const bf16x8*>(k_row + (r * D + 32 * dk + 8 * g));
      if (DK_TAIL) k_tail[b] = *reinterpret_cast<const shortx4*>(k_row + (r * D + (D - 16) + 4 * g));
      v_from[b] = v_cache + page_base + offset;
    }
#pragma unroll
    for (int b = 0; b < DC_BLOCKS; ++b)
#pragma unroll
      for (int db = 0; db < DB16; ++db)
        v_reg[b][db] = *reinterpret_cast<const uint2*>(v_from[b] + static_cast<int64_t>(16 * db) * block_size + (r * block_size + 4 * g));
    __builtin_amdgcn_sched_barrier(0);
    // the next chunk's pages, while this chunk's keys and values are on their way
    if (chunk + DC_KEYS <= key_end) {
#pragma unroll
      for (int b = 0; b < DC_BLOCKS; ++b)
        pages[b] = table[min((chunk + DC_KEYS + 16 * b) / block_size, table_width - 1)];
    }
    // ---- scores
    floatx4 s[MB][DC_BLOCKS];
#pragma unroll
    for (int b = 0; b < DC_BLOCKS; ++b) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) s[mb][b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dk = 0; dk < DK32; ++dk)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          s[mb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k_reg[b][dk], q_reg[mb][dk], s[mb][b], 0, 0, 0);
      if (DK_TAIL) {
        // The last 16 dims go through the 16-deep instruction into an accumulator of their own, added on the
        // vector ALU: chained straight onto the 32-deep instruction's accumulator, the first two of its
        // four registers were read before they were written (results depended on timing).
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const floatx4 tail = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(k_tail[b], q_tail[mb], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[mb][b][i] += tail[i];
        }
      }
    }
    // ---- softmax step per column
    bf16x8 p_reg[MB][DC_BLOCKS / 2];
    float alpha[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float best = -INFINITY;
#pragma unroll
      for (int b = 0; b < DC_BLOCKS; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = chunk + 16 * b + 4 * g + i;
          const float v = (key >= key_begin && key <= key_end) ? s[mb][b][i] * scale_log2 : -INFINITY;
          s[mb][b][i] = v;
          best = fmaxf(best, v);
        }
      best = lanes_max<16>(best);
      best = lanes_max<32>(best);
      const float m_new = fmaxf(m_run[mb], best);      // finite: every chunk of the run holds a key
      alpha[mb] = fast_exp2(m_run[mb] - m_new);        // 0 while m_run is -inf
      float sum = 0.f;
#pragma unroll
      for (int b = 0; b < DC_BLOCKS; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = fast_exp2(s[mb][b][i] - m_new);
          sum += p;
          p_reg[mb][b / 2][4 * (b % 2) + i] = static_cast<bf16_t>(p);
        }
      l_run[mb] = l_run[mb] * alpha[mb] + sum;      // the lanes of a column each keep a part of the sum
      m_run[mb] = m_new;
    }
    // ---- rescale what is there; the lane holds columns 4g..4g+3 of each output block
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float a4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a4[i] = __shfl(alpha[mb], 4 * g + i, DISTIE_WAVE);
#pragma unroll
      for (int db = 0; db < DB16; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) o_acc[mb][db][i] *= a4[i];
    }
    // Slots after the run's last key were never written by this request: what a former owner of the page left there must not
    // even be multiplied by a weight of zero (0 * NaN), so those values are cleared, and those of blocks outside the run. (Here and
    // not where they are loaded: there each block's values would be waited for before the next block's are asked for.)
    if (chunk < key_begin || chunk + DC_KEYS - 1 > key_end) {
#pragma unroll
      for (int b = 0; b < DC_BLOCKS; ++b) {
        const int written = b < low ? 0 : key_end - (chunk + 16 * b + 4 * g) + 1;          // of this lane's four keys
        const uint32_t keep_lo = written >= 2 ? 0xffffffffu : (written == 1 ? 0x0000ffffu : 0u);
        const uint32_t keep_hi = written >= 4 ? 0xffffffffu : (written == 3 ? 0x0000ffffu : 0u);
#pragma unroll
        for (int db = 0; db < DB16; ++db) v_reg[b][db].x &= keep_lo, v_reg[b][db].y &= keep_hi;
      }
    }
    // ---- O += P . V, 32 keys (two blocks) a step; the vector is put together as whole 32-bit words
#pragma unroll
    for (int ks = 0; ks < DC_BLOCKS / 2; ++ks)
#pragma unroll
      for (int db = 0; db < DB16; ++db) {
        const uintx4 words = {v_reg[2 * ks][db].x, v_reg[2 * ks][db].y, v_reg[2 * ks + 1][db].x, v_reg[2 * ks + 1][db].y};
        const bf16x8 v = __builtin_bit_cast(bf16x8, words);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          o_acc[mb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_reg[mb][ks], v, o_acc[mb][db], 0, 0, 0);
      }
  }

  // ---- sums over the lanes of a column, then the partial result of this run
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    l_run[mb] = lanes_sum<16>(l_run[mb]);
    l_run[mb] = lanes_sum<32>(l_run[mb]);
  }
  const int places = (max_splits + W - 1) / W;                  // for partial results, per request and head
  const int64_t head0 = static_cast<int64_t>(request) * heads + kh * group;
  // W > 1: sums [W][group][D], then maxima and sums of weights [W][group][2]
  extern __shared__ __attribute__((aligned(16))) float decode_lds[];
  float* ml_lds = decode_lds + W * group * D;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 16 * mb + 4 * g + i;
      const float l_col = __shfl(l_run[mb], 4 * g + i, DISTIE_WAVE);
      const float m_col = __shfl(m_run[mb], 4 * g + i, DISTIE_WAVE);
      if (col >= group) continue;
      const int64_t slot = W > 1 ? wave * group + col : (head0 + col) * max_splits + run;
      float* po = (W > 1 ? decode_lds : part_o) + slot * D;
      float* ml = (W > 1 ? ml_lds : part_ml) + 2 * slot;
#pragma unroll
      for (int db = 0; db < DB16; ++db) po[16 * db + r] = o_acc[mb][db][i];
      if (r == 0) {
        ml[0] = m_col;
        ml[1] = l_col;
      }
    }
  if constexpr (W > 1) {
    // the workgroup's runs in their order, four dims of a column a thread
    __syncthreads();
    for (int idx = threadIdx.x; idx < group * (D / 4); idx += DISTIE_WAVE * W) {
      const int col = idx / (D / 4), d = 4 * (idx % (D / 4));
      float m = -INFINITY;
#pragma unroll
      for (int v = 0; v < W; ++v) m = fmaxf(m, ml_lds[2 * (v * group + col)]);      // finite: the first wave holds a key
      float l = 0.f;
      float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < W; ++v) {
        const float weight = fast_exp2(ml_lds[2 * (v * group + col)] - m);        // 0 for a wave without a key, whose sums are 0
        l = fmaf(weight, ml_lds[2 * (v * group + col) + 1], l);
        const float4 o = *reinterpret_cast<const float4*>(decode_lds + (v * group + col) * D + d);
        sum.x = fmaf(weight, o.x, sum.x);
        sum.y = fmaf(weight, o.y, sum.y);
        sum.z = fmaf(weight, o.z, sum.z);
        sum.w = fmaf(weight, o.w, sum.w);
      }
      const int64_t slot = (head0 + col) * places + share;
      *reinterpret_cast<float4*>(part_o + slot * D + d) = sum;
      if (d == 0) {
        part_ml[2 * slot] = m;
        part_ml[2 * slot + 1] = l;
      }
    }
  }
}

// Combines the partial results of the runs of keys of one (request, head): grid (heads, requests), four waves.
// The maximum and the weight of every run are found first; then each wave adds a quarter of the runs (in order) for the output
// dims its lanes own, and the four sums are added in order through LDS. What bounds it is its chain: with weights through LDS
// (three barriers, a branch and a read of LDS a run) steps took, us, so / now: one request of 500 keys 1,076 / 1,049, 8 of 2,048 1,344 / 1,315,
// 64 of 2,048 2,339 / 2,318, 4 of 16,000 1,571 / 1,523.
// FAST (at most RD_FAST_RUNS runs fit the buffers): every partial result the block may need is asked for at
// once, before the request's length says which runs exist (their places are inside the buffers either way,
// and what a run that does not exist left there is dropped by a select, never multiplied): one trip to
// memory instead of three.
constexpr int RD_WAVES = 4;
constexpr int RD_THREADS = RD_WAVES * DISTIE_WAVE;
constexpr int RD_MAX_RUNS = 1024;
constexpr int RD_FAST_PER_WAVE = 16;
constexpr int RD_FAST_RUNS = RD_FAST_PER_WAVE * RD_WAVES;
static_assert(RD_FAST_RUNS == DISTIE_WAVE, "a lane a run");

template <bool FAST>
__global__ __launch_bounds__(RD_THREADS) void attn_reduce_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int32_t* __restrict__ kv_len,
    const int32_t* __restrict__ cu_q, bf16_t* __restrict__ out, int heads, int window, int all_splits, int together,
    int dense_rows, const int32_t* __restrict__ shared_run_len, const float* __restrict__ sinks) {
  const int max_splits = (all_splits + together - 1) / together;      // places: the runs of a workgroup share one
  __shared__ float weight_s[FAST ? 1 : RD_MAX_RUNS];
  __shared__ float sum_s[RD_WAVES][D];
  __shared__ float scratch[32];
  const int tid = threadIdx.x;
  const int wave = tid / DISTIE_WAVE;
  const int lane = tid % DISTIE_WAVE;
  const int request = blockIdx.y;
  const int head = blockIdx.x;
  const int64_t base0 = (static_cast<int64_t>(request) * heads + head) * max_splits;

  const int length = kv_len[request];
  const int run_len = shared_run_len != nullptr ? *shared_run_len : 0;
  float early[FAST ? RD_FAST_PER_WAVE : 1][DIMS_PER_LANE];
  float2 early_ml = {0.f, 0.f};
  if constexpr (FAST) {
    early_ml = *reinterpret_cast<const float2*>(part_ml + 2 * (base0 + min(lane, max_splits - 1)));
#pragma unroll
    for (int u = 0; u < RD_FAST_PER_WAVE; ++u) {
      const int j = min(wave + RD_WAVES * u, max_splits - 1);
#pragma unroll
      for (int i = 0; i < DIMS_PER_LANE; ++i) early[u][i] = part_o[(base0 + j) * D + min(lane + i * DISTIE_WAVE, D - 1)];
    }
    asm volatile("" ::"s"(length), "s"(run_len));           // (asked for here, not behind the branch below)
  }

  const int token = dense_rows ? request : cu_q[request];
  if (!dense_rows && cu_q[request + 1] - token != 1) return;
  const int q_pos = length - 1;
  const int all_runs = key_runs(q_pos, window, all_splits, run_len).count;
  const int runs = (all_runs + together - 1) / together;     // the first `runs` places hold results
  const int64_t base = base0;
  bf16_t* o = out + (static_cast<int64_t>(token) * heads + head) * D;
  // a sink: one more maximum and one more term of the denominator, in the runs' units of log 2; it has no value
  const float sink = sinks != nullptr ? sinks[head] * 1.4426950408889634f : -INFINITY;

  if constexpr (FAST) {
    // Every wave has all runs' maxima and sums in its lanes (RD_FAST_RUNS is a wave), and takes its own runs' weights from there: no
    // barrier and no trip to LDS but the one that puts the waves together.
    const bool mine = lane < runs;
    const float m = fmaxf(wave_max(mine ? early_ml.x : -INFINITY), sink);
    const float w = mine ? fast_exp2(early_ml.x - m) : 0.f;
    const float l = wave_sum(mine ? w * early_ml.y : 0.f) + (sink == -INFINITY ? 0.f : fast_exp2(sink - m));
    const int own = __builtin_amdgcn_readfirstlane(wave);
    float a[DIMS_PER_LANE] = {};
#pragma unroll
    for (int u = 0; u < RD_FAST_PER_WAVE; ++u) {
      const int j = own + RD_WAVES * u;
      const float weight = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), j));
#pragma unroll
      for (int i = 0; i < DIMS_PER_LANE; ++i) a[i] = j < runs ? fmaf(weight, early[u][i], a[i]) : a[i];
    }
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d < D) sum_s[wave][d] = a[i];
    }
    __syncthreads();
    if (wave != 0) return;
    const float inv = 1.f / l;
#pragma unroll
    for (int i = 0; i < DIMS_PER_LANE; ++i) {
      const int d = lane + i * DISTIE_WAVE;
      if (d < D) o[d] = static_cast<bf16_t>((((sum_s[0][d] + sum_s[1][d]) + sum_s[2][d]) + sum_s[3][d]) * inv);
    }
    return;
  }

  // the maximum over all runs (in units of log 2), then every run's weight
  float m = -INFINITY;
  for (int j = tid; j < runs; j += RD_THREADS) m = fmaxf(m, part_ml[2 * (base + j)]);
  m = wave_max(m);
  if (lane == 0) scratch[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3])), sink);
  float l = 0.f;
  for (int j = tid; j < runs; j += RD_THREADS) {
    const float w = fast_exp2(part_ml[2 * (base + j)] - m);
    weight_s[j] = w;
    l += w * part_ml[2 * (base + j) + 1];
  }
  l = block_sum(l, scratch + 16);           // has the barrier that publishes the weights
  if (sink != -INFINITY) l += fast_exp2(sink - m);
  const float* po = part_o + base * D;
#pragma unroll
  for (int i = 0; i < DIMS_PER_LANE; ++i) {
    const int d = lane + i * DISTIE_WAVE;
    if (d >= D) continue;
    float a = 0.f;
    int j = wave;
    for (; j + 3 * RD_WAVES < runs; j += 4 * RD_WAVES) {
      const float v0 = po[static_cast<int64_t>(j) * D + d], v1 = po[static_cast<int64_t>(j + RD_WAVES) * D + d];
      const float v2 = po[static_cast<int64_t>(j + 2 * RD_WAVES) * D + d], v3 = po[static_cast<int64_t>(j + 3 * RD_WAVES) * D + d];
      a = fmaf(weight_s[j], v0, a);
      a = fmaf(weight_s[j + RD_WAVES], v1, a);
      a = fmaf(weight_s[j + 2 * RD_WAVES], v2, a);
      a = fmaf(weight_s[j + 3 * RD_WAVES], v3, a);
    }
    for (; j < runs; j += RD_WAVES) a = fmaf(weight_s[j], po[static_cast<int64_t>(j) * D + d], a);
    sum_s[wave][d] = a;
  }
  __syncthreads();
  if (wave != 0) return;
  const float inv = 1.f / l;
#pragma unroll
  for (int i = 0; i < DIMS_PER_LANE; ++i) {
    const int d = lane + i * DISTIE_WAVE;
    if (d < D) o[d] = static_cast<bf16_t>((((sum_s[0][d] + sum_s[1][d]) + sum_s[2][d]) + sum_s[3][d]) * inv);
  }
}

// How many consecutive runs a workgroup puts together, one a wave. 1 as a rule: waves of their own spread best over the
// chip (8 of them in a workgroup read through one CU: 28 layers, 12 heads on 2, 1 request of 500 keys 1,442 -> 1,537 us,
// 8 of 2,048 keys 1,577 -> 1,645, 64 of 2,048 keys 2,580 -> 2,640). More than RD_FAST_RUNS partial results, though, cost the
// reduce 8.9 us a layer instead of 4.6, trip after trip to memory: put together they fit it. By 4 while those workgroups
// have a compute unit each, by 8 beyond; us a layer apart, by 4, by 8 (both kernels): 12 heads of 128 on 2, 1 request of
// 16,500 keys 15.0, 13.5, 18.7, of 65,000 28.6, 21.9, 30.1; 4 of 8,000 keys 16.4, 11.2, 13.9; 3 of 16,000 keys (378 workgroups
// by 4) 24.7, 15.2, 14.5; 28 on 4, 2 of 8,000 keys (256 workgroups) 16.6, 11.2, 13.9, 2 of 20,000 24.7, 20.7, 19.8.
// Of 240 steps (1 to 4 requests of 4,500 to 65,000 keys, heads of 32 to 256) this is at most 7 % from the best of the three and 2 % from runs apart.
// By 4 also for heads whose sums would fill the LDS. pairs: (request, kv head) pairs.
constexpr size_t DECODE_LDS = 64 * 1024;
constexpr int DECODE_MOST_TOGETHER = D <= 128 ? 8 : 4;        // more than 256 registers a wave: one wave a SIMD
extern "C" int distie_attention_decode_together(int max_splits, int group, int pairs) {
  if (max_splits <= RD_FAST_RUNS || group > 16) return 1;
  const bool by_four = (max_splits + 3) / 4 <= RD_FAST_RUNS && static_cast<int64_t>((max_splits + 3) / 4) * pairs <= 256;
  for (int together = by_four ? 4 : DECODE_MOST_TOGETHER; together >= 4; together /= 2)
    if (static_cast<size_t>(together) * group * (D + 2) * sizeof(float) <= DECODE_LDS) return together;
  return 1;
}

constexpr int DECODE_MAX_MB = (D <= 128) ? 4 : 2;   // registers: the output tile is 16 * MB x D floats a wave

// most query heads per kv head the decode kernel takes
extern "C" int distie_attention_decode_columns() { return 16 * DECODE_MAX_MB; }

// The requests of a step that bring one token (others are skipped). kv_len: tokens cached after the step, per
// request. part_o: float32 [requests, heads, max_splits, D], part_ml: float32 [requests, heads, max_splits, 2]:
// every request's keys are cut into at most max_splits runs by its own length. split_hint, a multiple of 64, is
// the run length the caller expects of the longest request; it only saves time where it is right.
// shared_run_len (no window, every request of the step brings one token; else null): int32 [1], one run length for
// all requests, with which no request has more than max_splits runs (distie_attention_decode_run_len).
extern "C" int distie_attention_decode_bf16(const void* qkv, int64_t q_stride, const void* k_cache, const void* v_cache,
                                            const int32_t* kv_len, const int32_t* cu_q, const int32_t* block_table,
                                            int table_width, const int32_t* table_rows, void* out, float* part_o, float* part_ml,
                                            int num_requests, int heads, int kv_heads, int block_size, float scale,
                                            int window, int split_hint, int max_splits, int dense_rows,
                                            const int32_t* shared_run_len, const float* sinks, int together,
                                            hipStream_t stream) {
  if (num_requests <= 0) return 0;
  const int group = kv_heads > 0 ? heads / kv_heads : 0;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || block_size % 16 != 0 || table_width < 1 ||
      split_hint < RUN_STEP || split_hint % RUN_STEP != 0 || max_splits < 1 || max_splits > RD_MAX_RUNS ||
      group > 16 * DECODE_MAX_MB || kv_heads > 65535 || num_requests > 65535 || heads > 65535 ||
      (shared_run_len != nullptr && (window != 0 || !dense_rows)))
    return DISTIE_BAD_ARGUMENT;
  const size_t lds = together > 1 ? static_cast<size_t>(together) * group * (D + 2) * sizeof(float) : 0;
  if ((together != 1 && together != 4 && together != DECODE_MOST_TOGETHER) || (together > 1 && group > 16) || lds > DECODE_LDS)
    return DISTIE_BAD_ARGUMENT;
  const int places = (max_splits + together - 1) / together;
  const dim3 grid = shared_run_len != nullptr ? dim3(kv_heads, num_requests, places) : dim3(places, kv_heads, num_requests);
  const bf16_t* q = static_cast<const bf16_t*>(qkv);
  const bf16_t* kc = static_cast<const bf16_t*>(k_cache);
  const bf16_t* vc = static_cast<const bf16_t*>(v_cache);
#define DECODE_LAUNCH(MB, W)                                                                                          \
  attn_decode_kernel<MB, W><<<grid, DISTIE_WAVE * W, lds, stream>>>(                                                   \
      q, q_stride, kc, vc, kv_len, cu_q, block_table, table_width, table_rows, part_o, part_ml, heads, kv_heads, block_size, \
      scale, window, split_hint, max_splits, dense_rows, shared_run_len)
  if (together == 4) {
    DECODE_LAUNCH(1, 4);
  } else if (together > 1) {
    DECODE_LAUNCH(1, DECODE_MOST_TOGETHER);
  } else if (group <= 16) {
    DECODE_LAUNCH(1, 1);
  } else if (group <= 32) {
    DECODE_LAUNCH(2, 1);
  } else {
    DECODE_LAUNCH(DECODE_MAX_MB, 1);
  }
#undef DECODE_LAUNCH
  int status = launch_status();
  if (status != 0) return status;
  if (places <= RD_FAST_RUNS) {
    attn_reduce_kernel<true><<<dim3(heads, num_requests), RD_THREADS, 0, stream>>>(
        part_o, part_ml, kv_len, cu_q, static_cast<bf16_t*>(out), heads, window, max_splits, together, dense_rows,
        shared_run_len, sinks);
  } else {
    attn_reduce_kernel<false><<<dim3(heads, num_requests), RD_THREADS, 0, stream>>>(
        part_o, part_ml, kv_len, cu_q, static_cast<bf16_t*>(out), heads, window, max_splits, together, dense_rows,
        shared_run_len, sinks);
  }
  return launch_status();
}

// ===================================================================================================
//  * attn_prefill: the tiled kernel for portions of prompts. A workgroup of four waves owns PF_BM
//    consecutive new tokens of one request and one head; it walks over the keys 64 at a time. The K tile
//    [64, D] and the V^T tile [D, 64] are put into LDS once per workgroup (global loads of the next tile
//    are in flight while the current one is used) and every wave multiplies its own 32 query columns
//    against them with the 32 x 32 x 16 products (per flop they read half the operands of the 16-wide ones,
//    which is what bounds those here):
//        S^T[key, col] = K[key, :] . q[col, :]     K rows from LDS as the A operand, q in registers
//        O^T[d, col]  += V^T[d, key] . P^T[key, col]
//    A lane holds, of a 32 x 32 score tile, keys 8i + 4h + j (i, j < 4) of column c (c = lane % 32,
//    h = lane / 32): so a lane's 32 scores of a key tile, its running maximum and sum and its 32 D / 64
//    output sums all belong to one query token, and nothing but the column's maximum moves between lanes.
//    The B operand of the second product wants 8 of 16 summed keys per lane: those are the lane's own
//    scores if the 16 keys of a step are taken in the order (4h..4h+3, 8+4h..8+4h+3), and V^T is read
//    from LDS in the same order.
//    Head sizes that are no multiple of 32 compute a last block of 32 output rows of which 16 are zeros.
//    Requests that bring fewer than `min_q_len` tokens are left to the decode kernel.
// ===================================================================================================
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
constexpr int PF_BN = 64;                               // keys per tile
constexpr int PF_WAVES = 4;
constexpr int PF_THREADS = PF_WAVES * DISTIE_WAVE;
constexpr int PF_WAVE_COLS = 32;
constexpr int PF_BM = PF_WAVES * PF_WAVE_COLS;          // query tokens per workgroup
constexpr float PF_GROW = 8.f;                          // in units of log 2: how far a score may pass a column's reference
constexpr int PF_DK = D / 16;                           // steps of the q.k product
constexpr int PF_DB = (D + 31) / 32;                    // blocks of 32 output rows
#ifndef DISTIE_PF_AHEAD
#define DISTIE_PF_AHEAD 6
#endif
constexpr int PF_AHEAD = DISTIE_PF_AHEAD;               // reads from LDS in flight ahead of the products
// Rows in LDS, in elements. A lane reads 16 bytes of row (lane % 32) of K, and two times 8 bytes of row
// (lane % 32) of V^T: free of bank conflicts when a row is an odd number of such pieces long (measured: K rows
// of 272 and 304 bytes read at 198 B/clk a compute unit, of 288 at 112; V^T rows of 136 bytes 207, of 144 116).
constexpr int PF_K_STRIDE = D + 8;
constexpr int PF_V_STRIDE = PF_BN + 4;
constexpr int PF_BLOCK_CHUNKS = 2 * D;                  // 16-byte pieces of 16 keys of K, and of V^T: [16, D] or [D, 16]
constexpr int PF_PASSES = (PF_BLOCK_CHUNKS + DISTIE_WAVE - 1) / DISTIE_WAVE;   // pieces a lane carries per block
static_assert(PF_WAVES * 16 == PF_BN, "each wave brings one block of 16 keys of a tile");

__global__ __launch_bounds__(PF_THREADS, (D <= 128) ? 2 : 1) void attn_prefill_kernel(
    const bf16_t* __restrict__ qkv, int64_t q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ positions, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows, bf16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int tokens, int num_requests, int heads, int kv_heads, int block_size, float scale,
    int window, int min_q_len, const float* __restrict__ sinks) {
  __shared__ __attribute__((aligned(16))) bf16_t k_lds[PF_BN * PF_K_STRIDE];
  __shared__ __attribute__((aligned(16))) bf16_t v_lds[32 * PF_DB * PF_V_STRIDE];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / DISTIE_WAVE);   // uniform: what depends on it alone stays scalar
  const int lane = tid % DISTIE_WAVE;
  const int c = lane % 32;
  const int h = lane / 32;
  const int group = heads / kv_heads;
  const float scale_log2 = scale * 1.4426950408889634f;      // scores in units of log 2: weights are exp2

  // ---- which tokens: tiles of PF_BM tokens over the requests that are served here, the last first: the late
  // tokens of a portion see the most keys, and the longest work should start first
  int tile = gridDim.y - 1 - blockIdx.y;
  int request = 0, begin = 0, end = 0;
  for (; request < num_requests; ++request) {
    begin = cu_q[request];
    end = cu_q[request + 1];
    if (end - begin < min_q_len) continue;
    const int tiles = (end - begin + PF_BM - 1) / PF_BM;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (request >= num_requests) return;
  const int head = blockIdx.x;                            // heads vary fastest: the heavy tiles of all heads start first
  const int kh = head / group;
  const int token0 = begin + tile * PF_BM;
  const int columns = min(PF_BM, end - token0);           // of the workgroup
  const int pos0 = positions[token0];                     // the tokens of a portion have consecutive positions
  const int key_begin = first_visible(pos0, window);
  const int key_end = pos0 + columns - 1;
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request] : request) * table_width;

  // the rows of V^T past the head size, read by the last block of output rows, stay zero
  if (D % 32 != 0)
    for (int i = tid; i < (32 * PF_DB - D) * PF_V_STRIDE; i += PF_THREADS) v_lds[D * PF_V_STRIDE + i] = static_cast<bf16_t>(0.f);

  // ---- this wave's columns; the lane's column
  const int wave_col0 = wave * PF_WAVE_COLS;
  const int wave_cols = max(0, min(PF_WAVE_COLS, columns - wave_col0));
  const int wave_last = pos0 + wave_col0 + wave_cols - 1;
  const int wave_first = first_visible(pos0 + wave_col0, window);
  const int wave_open = first_visible(max(wave_last, 0), window);      // from here on every column of the wave sees (up to its own position)
  const int col = min(wave_col0 + c, columns - 1);        // columns past the end repeat the last; dropped later
  const int col_last = pos0 + col;                        // the last key the column sees, and the first
  const int col_first = first_visible(col_last, window);
  bf16x8 q_reg[PF_DK];
  {
    const bf16_t* q = qkv + (token0 + col) * q_stride + static_cast<int64_t>(head) * D;
#pragma unroll
    for (int dk = 0; dk < PF_DK; ++dk) q_reg[dk] = *reinterpret_cast<const bf16x8*>(q + 16 * dk + 8 * h);
  }
  floatx16 o_acc[PF_DB];
#pragma unroll
  for (int db = 0; db < PF_DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o_acc[db][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // ---- staging of one tile in registers. Wave w brings block w of the tile (keys k0 + 16 w .. + 15): one page
  // lookup a wave, the 16 rows of K are one run of 16 D elements in their page, V^T is D runs of 16.
  uint4 k_stage[PF_PASSES], v_stage[PF_PASSES];
  const int block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  // Every lane issues the same loads for every tile, with no branch around them: a block that belongs to no
  // page reads the start of the cache instead and is cleared when it is stored.
  auto block_live = [&](int key) { return key <= key_end && key + 15 >= key_begin; };
  // The page of a block is looked up two tiles before its keys are asked for (a scalar load, the block being
  // the same for the whole wave): asked for together, every tile would cost the wave two trips to memory
  // one after the other.
  auto lookup = [&](int k0) {
    const int key = k0 + 16 * wave;
    const int slot = block_shift >= 0 ? key >> block_shift : key / block_size;
    return table[min(slot, table_width - 1)];
  };
  auto fetch = [&](int k0, int page_of_block) {
    const int key = k0 + 16 * wave;
    const bool live = block_live(key);
    const int offset = live ? (block_shift >= 0 ? key & (block_size - 1) : key % block_size) : 0;
    const int page = live ? page_of_block : 0;
    const int64_t base = live ? (static_cast<int64_t>(page) * kv_heads + kh) * block_size * D : 0;
    const bf16_t* k_block = k_cache + base + static_cast<int64_t>(offset) * D;
    const bf16_t* v_block = v_cache + base + offset;
#pragma unroll
    for (int p = 0; p < PF_PASSES; ++p) {
      const int j = min(lane + p * DISTIE_WAVE, PF_BLOCK_CHUNKS - 1);
      k_stage[p] = *reinterpret_cast<const uint4*>(k_block + 8 * j);
      v_stage[p] = *reinterpret_cast<const uint4*>(v_block + static_cast<int64_t>(j / 2) * block_size + 8 * (j % 2));
    }
  };
  // where a lane's pieces go in LDS: the same for every tile (a row of V^T is a multiple of 8 bytes long,
  // not of 16: its pieces are stored as two halves)
  int k_slot[PF_PASSES], v_slot[PF_PASSES];
#pragma unroll
  for (int p = 0; p < PF_PASSES; ++p) {
    const int j = min(lane + p * DISTIE_WAVE, PF_BLOCK_CHUNKS - 1);
    k_slot[p] = (16 * wave + j / (D / 8)) * PF_K_STRIDE + 8 * (j % (D / 8));
    v_slot[p] = (j / 2) * PF_V_STRIDE + 16 * wave + 8 * (j % 2);
  }
  auto stash = [&](int k0) {
    const int key = k0 + 16 * wave;                       // the same for the whole wave: the branches are uniform
    const bool live = block_live(key);
    // Slots after the last key of this workgroup were not written by this request, and blocks outside the keys
    // of this workgroup were not read: cleared (a weight of zero times NaN would still be NaN).
    const bool whole = live && key + 15 <= key_end;
    if (whole) {
#pragma unroll
      for (int p = 0; p < PF_PASSES; ++p) {
        if (lane + p * DISTIE_WAVE >= PF_BLOCK_CHUNKS) continue;
        *reinterpret_cast<uint4*>(k_lds + k_slot[p]) = k_stage[p];
        *reinterpret_cast<uint2*>(v_lds + v_slot[p]) = uint2{v_stage[p].x, v_stage[p].y};
        *reinterpret_cast<uint2*>(v_lds + v_slot[p] + 4) = uint2{v_stage[p].z, v_stage[p].w};
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < PF_PASSES; ++p) {
      const int j = lane + p * DISTIE_WAVE;
      if (j >= PF_BLOCK_CHUNKS) continue;
      *reinterpret_cast<uint4*>(k_lds + k_slot[p]) = live ? k_stage[p] : uint4{0u, 0u, 0u, 0u};
      const int written = live ? key_end - (key + 8 * (j % 2)) + 1 : 0;        // of this piece's eight keys
      const uint32_t w[4] = {v_stage[p].x, v_stage[p].y, v_stage[p].z, v_stage[p].w};
      uint32_t m[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m[e] = written >= 2 * e + 2 ? w[e] : (written == 2 * e + 1 ? (w[e] & 0x0000ffffu) : 0u);
      *reinterpret_cast<uint2*>(v_lds + v_slot[p]) = uint2{m[0], m[1]};
      *reinterpret_cast<uint2*>(v_lds + v_slot[p] + 4) = uint2{m[2], m[3]};
    }
  };

  auto compute = [&](int k0) {
    if (wave_cols <= 0 || k0 > wave_last || k0 + PF_BN - 1 < wave_first) return;

    // ---- scores: 64 keys x the wave's 32 columns, as two blocks of 32 keys
    floatx16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kb][e] = 0.f;
    // PF_AHEAD reads from LDS are under way when the first product is issued, and every product is followed
    // by one more read: left to itself the compiler keeps two reads in flight, which is less than the trip takes
    {
      bf16x8 a[2 * PF_DK];
#pragma unroll
      for (int i = 0; i < 2 * PF_DK; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(k_lds + (32 * (i % 2) + c) * PF_K_STRIDE + 16 * (i / 2) + 8 * h);
#pragma unroll
      for (int i = 0; i < 2 * PF_DK; ++i)
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], q_reg[i / 2], s[i % 2], 0, 0, 0);
      constexpr int ahead = 2 * PF_DK < PF_AHEAD ? 2 * PF_DK : PF_AHEAD;
      __builtin_amdgcn_sched_group_barrier(0x100, ahead, 0);
#pragma unroll
      for (int i = 0; i < 2 * PF_DK - ahead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, ahead, 0);
    }
    // ---- softmax step of the lane's column. A tile whose keys every column of the wave sees needs no mask:
    // that is every tile but those on the diagonal and at a window's edge.
    const bool tile_open = k0 + PF_BN - 1 <= pos0 + wave_col0 &&
                           k0 >= wave_open;
    if (!tile_open) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = k0 + 32 * kb + 8 * (e / 4) + 4 * h + e % 4;
          if (key < col_first || key > col_last) s[kb][e] = -INFINITY;
        }
    }
    // The running reference m of a column (scores count from it: weights are 2^(score - m)) follows the
    // largest score only when that has grown by more than PF_GROW since m was set: then the sums so far are
    // scaled down, for all columns of the wave at once. In between a weight may reach 2^PF_GROW, which
    // float32 sums and bfloat16 weights hold as well as they hold 1, and the scaling of the sums becomes rare.
    float top = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) top = fmaxf(top, s[kb][e]);
    top = lanes_max<32>(top);
    const float best = top * scale_log2;                  // the scale is positive: the largest stays the largest
    if (__any(best > m_run + PF_GROW)) {                  // also the first score of a column (m = -inf)
      const float m_new = fmaxf(m_run, best);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);   // 0 while m was -inf
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int db = 0; db < PF_DB; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o_acc[db][e] *= alpha;
    }
    const float from = m_run == -INFINITY ? 0.f : -m_run;
    bf16x8 p_reg[4];                                      // step t: keys 16 t + (4h..4h+3, 8+4h..8+4h+3) of the tile
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = fast_exp2(fmaf(s[kb][e], scale_log2, from));
        sum += p;
        p_reg[2 * kb + e / 8][e % 8] = static_cast<bf16_t>(p);
      }
    l_run += sum;
    // ---- O^T += V^T . P^T: four steps of 16 keys
    {
      bf16x8 vt[4 * PF_DB];
#pragma unroll
      for (int i = 0; i < 4 * PF_DB; ++i) {
        const bf16_t* v_row = v_lds + (32 * (i % PF_DB) + c) * PF_V_STRIDE + 16 * (i / PF_DB) + 4 * h;
        const uint2 lo = *reinterpret_cast<const uint2*>(v_row);
        const uint2 hi = *reinterpret_cast<const uint2*>(v_row + 8);
        const uintx4 words = {lo.x, lo.y, hi.x, hi.y};
        vt[i] = __builtin_bit_cast(bf16x8, words);
      }
#pragma unroll
      for (int i = 0; i < 4 * PF_DB; ++i)
        o_acc[i % PF_DB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vt[i], p_reg[i / PF_DB], o_acc[i % PF_DB], 0, 0, 0);
      constexpr int ahead = 4 * PF_DB < PF_AHEAD ? 4 * PF_DB : PF_AHEAD;
      __builtin_amdgcn_sched_group_barrier(0x100, ahead, 1);
#pragma unroll
      for (int i = 0; i < 4 * PF_DB - ahead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, ahead, 1);
    }
  };

  // With gridDim.z > 1 the key tiles of these tokens are cut in that many parts, one workgroup each, which write
  // unnormalised partial results that attn_prefill_merge_kernel combines: the last tokens of a long
  // portion walk over many key tiles one after the other, and this shortens the longest walk.
  // One tile of loads is in flight (tiles past the last key load the start of the cache and are not used).
  const int all_tile0 = key_begin / PF_BN * PF_BN;
  const int all_tiles = (key_end - all_tile0) / PF_BN + 1;
  const int per_split = (all_tiles + gridDim.z - 1) / gridDim.z;
  const int tile0 = all_tile0 + static_cast<int>(blockIdx.z) * per_split * PF_BN;
  const int loop_end = min(key_end, tile0 + per_split * PF_BN - 1);            // last key of this workgroup's walk
  fetch(tile0, lookup(tile0));
  int page_ahead = lookup(tile0 + PF_BN);
  for (int k0 = tile0; k0 <= loop_end; k0 += PF_BN) {
    __syncthreads();                       // every wave is done with the tile in LDS
    stash(k0);
    __syncthreads();
    fetch(k0 + PF_BN, page_ahead);
    page_ahead = lookup(k0 + 2 * PF_BN);
    compute(k0);
  }
  // ---- write: the lane holds, of its column, output rows 32 db + 8 i + 4 h + (0..3)
  l_run = lanes_sum<32>(l_run);
  if (wave_col0 + c >= columns) return;
  const int64_t row = static_cast<int64_t>(token0 + wave_col0 + c) * heads + head;
  if (gridDim.z == 1) {
    bf16_t* o = out + row * D;
    const float inv = sink_factor(m_run, l_run, sinks != nullptr ? sinks[head] * 1.4426950408889634f : -INFINITY);
#pragma unroll
    for (int db = 0; db < PF_DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 32 * db + 8 * i + 4 * h;
        if (d >= D) continue;
        uint32_t half[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) half[j] = __builtin_bit_cast(uint16_t, static_cast<bf16_t>(o_acc[db][4 * i + j] * inv));
        *reinterpret_cast<uint2*>(o + d) = uint2{half[0] | (half[1] << 16), half[2] | (half[3] << 16)};
      }
  } else {
    // a part without a key for this column leaves l = 0, and the merge does not read its sums
    const int64_t at = static_cast<int64_t>(blockIdx.z) * tokens * heads + row;
    float* po = part_o + at * D;
#pragma unroll
    for (int db = 0; db < PF_DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 32 * db + 8 * i + 4 * h;
        if (d >= D) continue;
        *reinterpret_cast<float4*>(po + d) = float4{o_acc[db][4 * i], o_acc[db][4 * i + 1], o_acc[db][4 * i + 2], o_acc[db][4 * i + 3]};
      }
    if (h == 0) {
      part_ml[2 * at] = m_run;
      part_ml[2 * at + 1] = l_run;
    }
  }
}

// Combines the `splits` parts of attn_prefill_kernel with gridDim.z > 1, in order: one block per token; tokens
// of requests that the kernel skipped (fewer than min_q_len tokens) are skipped here as well.
constexpr int PF_MAX_SPLITS = 16;

template <typename OUT, int MOST>
__global__ void attn_prefill_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                          const int32_t* __restrict__ token_request, const int32_t* __restrict__ cu_q,
                                          OUT* __restrict__ out, int tokens, int heads, int min_q_len, int splits,
                                          const float* __restrict__ sinks) {
  const int64_t token = blockIdx.x;
  const int request = token_request[token];
  if (cu_q[request + 1] - cu_q[request] < min_q_len) return;
  const int64_t part = static_cast<int64_t>(tokens) * heads;
  for (int i = threadIdx.x; i < heads * (D / 4); i += blockDim.x) {
    const int head = i / (D / 4);
    const int d = 4 * (i % (D / 4));
    const int64_t row = token * heads + head;
    float2 ml[MOST];
    float4 o[MOST];
    float m = -INFINITY;
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
      ml[s] = float2{-INFINITY, 0.f};
      o[s] = float4{0.f, 0.f, 0.f, 0.f};
      if (s < splits) ml[s] = *reinterpret_cast<const float2*>(part_ml + 2 * (s * part + row));
      // a part without a key for this token has l = 0; what it left in part_o is not read (for a prompt
      // without a past that is a third of all reads: asking for them anyway, to save the second trip to
      // memory, made this kernel slower where it runs, 12.2 -> 14.7 us, and 10.0 -> 10.5 once the registers of
      // the parts that are not there no longer held waves back)
      if (s < splits && ml[s].y > 0.f) {
        o[s] = *reinterpret_cast<const float4*>(part_o + (s * part + row) * D + d);
        m = fmaxf(m, ml[s].x);
      }
    }
    // a sink: one more maximum and one more term of the denominator, without a value
    const float sink = sinks != nullptr ? sinks[head] * 1.4426950408889634f : -INFINITY;
    m = fmaxf(m, sink);
    float l = sink == -INFINITY ? 0.f : fast_exp2(sink - m);
    float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
      const float w = ml[s].y > 0.f ? fast_exp2(ml[s].x - m) : 0.f;
      l += w * ml[s].y;
      sum.x += w * o[s].x;
      sum.y += w * o[s].y;
      sum.z += w * o[s].z;
      sum.w += w * o[s].w;
    }
    const float inv = 1.f / l;
    const float v[4] = {sum.x * inv, sum.y * inv, sum.z * inv, sum.w * inv};
    if constexpr (sizeof(OUT) == 4) {
      *reinterpret_cast<float4*>(out + row * D + d) = float4{v[0], v[1], v[2], v[3]};
    } else {
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = __builtin_bit_cast(uint16_t, static_cast<bf16_t>(v[e]));
      *reinterpret_cast<uint2*>(out + row * D + d) = uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
  }
}

// The merge holds every part's maximum, sum and four outputs in registers: compiled for at most 4, 8 and 16 parts,
// so that few parts leave room for more waves on a compute unit.
template <typename OUT>
static void launch_merge(const float* part_o, const float* part_ml, const int32_t* token_request, const int32_t* cu_q,
                         OUT* out, int tokens, int heads, int min_q_len, int splits, const float* sinks,
                         hipStream_t stream) {
  const int work = heads * (D / 4);
  const int threads = work >= 512 ? 512 : (work >= 256 ? 256 : 64);
  if (splits <= 4)
    attn_prefill_merge_kernel<OUT, 4><<<tokens, threads, 0, stream>>>(part_o, part_ml, token_request, cu_q, out, tokens,
                                                                       heads, min_q_len, splits, sinks);
  else if (splits <= 8)
    attn_prefill_merge_kernel<OUT, 8><<<tokens, threads, 0, stream>>>(part_o, part_ml, token_request, cu_q, out, tokens,
                                                                       heads, min_q_len, splits, sinks);
  else
    attn_prefill_merge_kernel<OUT, PF_MAX_SPLITS><<<tokens, threads, 0, stream>>>(part_o, part_ml, token_request, cu_q, out,
                                                                                   tokens, heads, min_q_len, splits, sinks);
}

// Portions of prompts (and whole mixed steps). bfloat16 only; block_size must be a multiple of 16. Requests that
// bring fewer than min_q_len tokens are skipped (the decode kernel serves them).
extern "C" int distie_attention_prefill_bf16(const void* qkv, int64_t q_stride, const void* k_cache, const void* v_cache,
                                             const int32_t* positions, const int32_t* cu_q, const int32_t* block_table,
                                             int table_width, const int32_t* table_rows, void* out, int tokens, int num_requests, int heads,
                                             int kv_heads, int block_size, float scale, int window, int min_q_len,
                                             const int32_t* token_request, float* part_o, float* part_ml,
                                             int splits, const float* sinks, hipStream_t stream) {
  // splits > 1: the keys are walked in that many parts side by side (worth it for long portions), with
  // part_o (float32 [splits, tokens, heads, D]) and part_ml (float32 [splits, tokens, heads, 2]) in between.
  if (tokens <= 0) return 0;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || block_size % 16 != 0 || table_width < 1 ||
      num_requests < 1 || heads > 65535 || min_q_len < 1 || splits < 1 || splits > PF_MAX_SPLITS || !(scale > 0.f) ||
      (splits > 1 && (part_o == nullptr || part_ml == nullptr || token_request == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const int tiles = (tokens + PF_BM - 1) / PF_BM + num_requests;     // an upper bound; spare blocks leave at once
  if (tiles > 65535) return DISTIE_BAD_ARGUMENT;
  attn_prefill_kernel<<<dim3(heads, tiles, splits), PF_THREADS, 0, stream>>>(
      static_cast<const bf16_t*>(qkv), q_stride, static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache),
      positions, cu_q, block_table, table_width, table_rows, static_cast<bf16_t*>(out), part_o, part_ml, tokens, num_requests, heads,
      kv_heads, block_size, scale, window, min_q_len, sinks);
  int status = launch_status();
  if (status != 0 || splits == 1) return status;
  launch_merge(part_o, part_ml, token_request, cu_q, static_cast<bf16_t*>(out), tokens, heads, min_q_len, splits, sinks, stream);
  return launch_status();
}

// ===================================================================================================
//  * attn_prefill_keys: the same products, cut the other way: the W waves of a workgroup share its 32 query columns (tokens of one
//    head) and each walks every W-th tile of 32 keys on its own. A wave's K and V^T tiles come from memory straight into a piece of
//    LDS of its own, the next ones while it multiplies the present ones, so the loop has no barrier; behind it the W sums
//    meet in LDS. A prompt of a few hundred tokens is one trip for q, K and V, one to three tiles a wave and that end, where
//    attn_prefill is a walk over all its keys by a fifth of the chip, and parts that a second launch merges.
//    K rows lie in LDS with their 16-byte pieces turned by the row's number (piece j of row r at j ^ r), which the loads
//    do and which keeps the reads of 32 rows free of bank conflicts; a row of V^T of 16 keys is two pieces, read in order. The
//    rows of a product are taken in an order in which a lane's scores are eight keys in a row, and those it reads of V^T.
//    12 heads of 128 and 2 kv heads, us, attn_prefill with its merge / this: 40 tokens 6.3 / 5.6, 301 13.5 / 7.7, 512 17.5 / 8.8, 1,024
//    27.2 / 14.0, 2,048 38.0 / 27.1. What bounds it: of the 5.6, 2 are the launch and the rest a chain of trips (requests, positions
//    and pages, keys, the sums); a tile costs a wave about 1 us alone on its SIMD and 1.3 beside another, a quarter of it products: reads
//    of LDS, the softmax and the next loads' addresses, one behind the other. Two waves a SIMD need the small tile: 64 keys at one wave
//    a SIMD 51 us for 2,048 tokens, 64 keys and 64 columns 42 (then 41 at 32 keys). The columns' maximum went through LDS at first, the
//    queries were waited for together with the first keys, and loads beyond the last tile were issued: 40 (W = 8), 32 (W = 4).
// ===================================================================================================
#if DISTIE_HEAD_DIM == 64 || DISTIE_HEAD_DIM == 128
constexpr int KEYS_BM = 32;                             // tokens of a workgroup
constexpr int KEYS_BN = 32;                             // keys of a wave's tile
constexpr int KEYS_PIECES = D / 8;                      // 16-byte pieces of a row of K
constexpr int KEYS_LOADS = D / 32;                      // loads (of 1 KB) of 16 keys of K, and of V^T
constexpr int KEYS_O_STRIDE = D + 4;                    // floats: rows of an odd number of 16-byte pieces

typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));

// LDS: the waves' tiles and, in their place, their sums; behind that their references and the columns' factors
template <int W>
constexpr int prefill_keys_tiles() {
  const int tiles = W * KEYS_BN * D * 4, sums = W * KEYS_BM * KEYS_O_STRIDE * 4;
  return tiles > sums ? tiles : sums;
}
template <int W>
constexpr int prefill_keys_lds() { return prefill_keys_tiles<W>() + (W + 1) * KEYS_BM * 8; }

template <int W>
__global__ __launch_bounds__(DISTIE_WAVE * W) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_prefill_keys_kernel(
    const bf16_t* __restrict__ qkv, int64_t q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ positions, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows, bf16_t* __restrict__ out,
    int num_requests, int heads, int kv_heads, int block_size, float scale, int window, int min_q_len,
    const float* __restrict__ sinks) {
  constexpr int BLOCKS = KEYS_BN / 16;
  constexpr int LOADS = BLOCKS * KEYS_LOADS;            // of a tile of K, and of V^T
  constexpr int STEP = W * KEYS_BN;
  extern __shared__ __attribute__((aligned(16))) char keys_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / DISTIE_WAVE);
  const int lane = threadIdx.x % DISTIE_WAVE;
  const int c = lane % 32;
  const int h = lane / 32;
  const float scale_log2 = scale * 1.4426950408889634f;

  // ---- which tokens: as attn_prefill, the late ones first
  int tile = gridDim.y - 1 - blockIdx.y;
  int request = 0, begin = 0, end = 0;
  for (; request < num_requests; ++request) {
    begin = cu_q[request];
    end = cu_q[request + 1];
    if (end - begin < min_q_len) continue;
    const int tiles = (end - begin + KEYS_BM - 1) / KEYS_BM;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (request >= num_requests) return;
  const int head = blockIdx.x;
  const int kh = head / (heads / kv_heads);
  const int token0 = begin + tile * KEYS_BM;
  const int columns = min(KEYS_BM, end - token0);
  const int pos0 = positions[token0];                   // the tokens of a portion have consecutive positions
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request] : request) * table_width;
  const int block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;

  // ---- the queries, on their way before anything says which keys they see
  const int col = min(c, columns - 1);                  // columns past the end repeat the last; dropped later
  bf16x8 q_reg[PF_DK];
  {
    const bf16_t* q = qkv + (token0 + col) * q_stride + static_cast<int64_t>(head) * D;
#pragma unroll
    for (int dk = 0; dk < PF_DK; ++dk) q_reg[dk] = *reinterpret_cast<const bf16x8*>(q + 16 * dk + 8 * h);
  }

  // ---- tiles into LDS
  char* const k_tile = keys_lds + wave * (KEYS_BN * D * 4);
  char* const v_tile = k_tile + KEYS_BN * D * 2;
  const uint32_t k_at = lds_place(k_tile), v_at = lds_place(v_tile);
  int k_lane[KEYS_LOADS], v_lane[KEYS_LOADS];
#pragma unroll
  for (int j = 0; j < KEYS_LOADS; ++j) {
    const int row = (DISTIE_WAVE / KEYS_PIECES) * j + lane / KEYS_PIECES;
    k_lane[j] = row * (2 * D) + ((lane % KEYS_PIECES) ^ (row % KEYS_PIECES)) * 16;
    const int piece = DISTIE_WAVE * j + lane;
    v_lane[j] = (piece / 2) * (2 * block_size) + (piece % 2) * 16;
  }
  struct Pages { int of[BLOCKS]; };
  auto lookup = [&](int k0) __attribute__((always_inline)) {
    Pages pages;
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
      const int key = k0 + 16 * b;
      const int slot = block_shift >= 0 ? key >> block_shift : key / block_size;
      pages.of[b] = table[min(slot, table_width - 1)];
    }
    return pages;
  };
  // A block of 16 keys outside the workgroup's keys belongs to no page that is known here: its loads read beyond the end of
  // an empty buffer, which gives zeros.
  int key_begin = 0, key_end = 0;
  const uint32_t page_bytes = 2u * static_cast<uint32_t>(kv_heads) * block_size * D;
  const char* const k_head = reinterpret_cast<const char*>(k_cache) + 2 * static_cast<int64_t>(kh) * block_size * D;
  const char* const v_head = reinterpret_cast<const char*>(v_cache) + 2 * static_cast<int64_t>(kh) * block_size * D;
  auto ask = [&](int k0, const Pages& pages, bool values) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
      const int key = k0 + 16 * b;
      const bool live = key <= key_end && key + 15 >= key_begin;
      const int offset = block_shift >= 0 ? key & (block_size - 1) : key % block_size;
      const uint64_t page = static_cast<uint64_t>(static_cast<uint32_t>(pages.of[b])) * page_bytes;
      if (values) {
        const intx4 from = buffer_of(v_head + page + 2 * offset, live ? 2 * ((D - 1) * block_size + 16) : 0);
#pragma unroll
        for (int j = 0; j < KEYS_LOADS; ++j) buffer_to_lds(from, v_lane[j], 0, v_at + (b * KEYS_LOADS + j) * 1024);
      } else {
        const intx4 from = buffer_of(k_head + page + 2 * D * offset, live ? 32 * D : 0);
#pragma unroll
        for (int j = 0; j < KEYS_LOADS; ++j) buffer_to_lds(from, k_lane[j], 0, k_at + (b * KEYS_LOADS + j) * 1024);
      }
    }
  };
  // (without a window the first pages do not wait for the position)
  int k0 = wave * KEYS_BN;
  if (window != 0) k0 += first_visible(pos0, window) / KEYS_BN * KEYS_BN;
  Pages pages = lookup(k0);
  key_begin = first_visible(pos0, window);
  key_end = pos0 + columns - 1;
  const int col_last = pos0 + col, col_first = first_visible(col_last, window);       // what the lane's column sees
  const int open_from = first_visible(key_end, window); // from here on every column sees (up to its own position)
  // (the queries are waited for here: a wait for them inside the loop would wait for its tiles as well)
#pragma unroll
  for (int dk = 0; dk < PF_DK; ++dk) asm volatile("" : "+v"(q_reg[dk]));
  if (k0 <= key_end) {
    ask(k0, pages, false);
    ask(k0, pages, true);
    if (k0 + STEP <= key_end) pages = lookup(k0 + STEP);
  }

  floatx16 o_acc[PF_DB];
#pragma unroll
  for (int db = 0; db < PF_DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o_acc[db][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  // the row of K behind row c of a product, and where its pieces are
  const int row = 16 * (c / 16) + 8 * ((c / 4) % 2) + 4 * ((c / 8) % 2) + c % 4;
  int piece_at[PF_DK];
#pragma unroll
  for (int dk = 0; dk < PF_DK; ++dk) piece_at[dk] = row * (2 * D) + ((2 * dk + h) ^ (row % KEYS_PIECES)) * 16;

  for (; k0 <= key_end; k0 += STEP) {
    const bool more = k0 + STEP <= key_end;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");       // K is there; V^T is under way
    floatx16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int dk = 0; dk < PF_DK; ++dk) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(k_tile + piece_at[dk]);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, q_reg[dk], s, 0, 0, 0);
    }
    // (all reads before the first product: left to itself the compiler keeps two under way)
    __builtin_amdgcn_sched_group_barrier(0x100, PF_DK, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, PF_DK, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // K has been read: its place is free
    if (more) ask(k0 + STEP, pages, false);

    if (k0 + KEYS_BN - 1 > pos0 || k0 < open_from) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = k0 + 16 * (e / 8) + 8 * h + e % 8;
        if (key < col_first || key > col_last) s[e] = -INFINITY;
      }
    }
    // the running reference follows the largest score as in attn_prefill
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) top = fmaxf(top, s[e]);
    const float best = lanes_max<32>(top) * scale_log2;
    if (__any(best > m_run + PF_GROW)) {
      const float m_new = fmaxf(m_run, best);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int db = 0; db < PF_DB; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o_acc[db][e] *= alpha;
    }
    const float from = m_run == -INFINITY ? 0.f : -m_run;
    bf16x8 p_reg[BLOCKS];                               // step t: keys 16 t + 8 h .. + 7 of the tile
#pragma unroll
    for (int e = 0; e < 16; ++e) p_reg[e / 8][e % 8] = static_cast<bf16_t>(fast_exp2(fmaf(s[e], scale_log2, from)));
    // What the weights are divided by is the sum of them as they go into the product: what rounding does to one that outdoes the
    // others cancels. Summed before they were rounded, the outputs of peaked scores (three units of spread) were further from 64 bits
    // than those of attn_prefill, whose references are found among more keys (1,024 tokens: W = 2 0.00205, W = 4 0.00196, attn_prefill
    // 0.00191; now 0.00186 and 0.00182). 1 to 3 % of the kernel: 2,048 tokens 26.5 -> 26.9 us, 301 7.63 -> 7.69.
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e += 2)
      sum = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{p_reg[e / 8][e % 8], p_reg[e / 8][e % 8 + 1]}, bf16x2{bf16_t(1.f), bf16_t(1.f)}, sum,
                                            false);
    l_run += sum;
    if (more)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");     // V^T is there; the next K is under way
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (k0 + KEYS_BN - 1 > key_end && key_end % 16 != 15) {
      // Slots after the last key were not written by this request (a weight of zero times NaN would still be NaN).
      const int b = (key_end - k0) / 16, left = key_end % 16 + 1;       // the block of the last key, and its keys
#pragma unroll
      for (int j = 0; j < KEYS_LOADS; ++j) {
        const int piece = DISTIE_WAVE * j + lane;
        const int written = left - 8 * (piece % 2);
        uint4* const at = reinterpret_cast<uint4*>(v_tile + b * (32 * D) + piece * 16);
        const uint4 v = *at;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        uint32_t m[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = written >= 2 * e + 2 ? w[e] : (written == 2 * e + 1 ? (w[e] & 0x0000ffffu) : 0u);
        *at = uint4{m[0], m[1], m[2], m[3]};
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int t = 0; t < BLOCKS; ++t)
#pragma unroll
      for (int db = 0; db < PF_DB; ++db) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(v_tile + t * (32 * D) + db * 1024 + (2 * c + h) * 16);
        o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, p_reg[t], o_acc[db], 0, 0, 0);
      }
    __builtin_amdgcn_sched_group_barrier(0x100, BLOCKS * PF_DB, 1);
    __builtin_amdgcn_sched_group_barrier(0x008, BLOCKS * PF_DB, 1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // V^T has been read
    if (more) {
      ask(k0 + STEP, pages, true);
      if (k0 + 2 * STEP <= key_end) pages = lookup(k0 + 2 * STEP);
    }
  }

  // ---- the waves' sums, put together: each scaled to the largest reference (a sink is one more), then added in order
  lds_arrived<0>();                                     // nothing under way, and every wave is done with its tiles
  float* const sums = reinterpret_cast<float*>(keys_lds);
  float2* const refs = reinterpret_cast<float2*>(keys_lds + prefill_keys_tiles<W>());     // [wave][column]
  float* const inverse = reinterpret_cast<float*>(refs + W * KEYS_BM);                    // [column]
  l_run = lanes_sum<32>(l_run);
  if (h == 0) refs[wave * KEYS_BM + c] = float2{m_run, l_run};
  __syncthreads();
  {
    const float sink = sinks != nullptr ? sinks[head] * 1.4426950408889634f : -INFINITY;
    float2 ml[W];
    float m = sink;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      ml[w] = refs[w * KEYS_BM + c];
      m = fmaxf(m, ml[w].x);
    }
    float l = sink == -INFINITY ? 0.f : fast_exp2(sink - m);
#pragma unroll
    for (int w = 0; w < W; ++w) l += ml[w].x == -INFINITY ? 0.f : fast_exp2(ml[w].x - m) * ml[w].y;
    if (wave == 0 && h == 0) inverse[c] = 1.f / l;
    const float alpha = m_run == -INFINITY ? 0.f : fast_exp2(m_run - m);
    float* const to = sums + (wave * KEYS_BM + c) * KEYS_O_STRIDE + 4 * h;
#pragma unroll
    for (int db = 0; db < PF_DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(to + 32 * db + 8 * i) = float4{o_acc[db][4 * i] * alpha, o_acc[db][4 * i + 1] * alpha,
                                                                 o_acc[db][4 * i + 2] * alpha, o_acc[db][4 * i + 3] * alpha};
  }
  __syncthreads();
  for (int i = threadIdx.x; i < columns * (D / 4); i += DISTIE_WAVE * W) {
    const int to = i / (D / 4), d = 4 * (i % (D / 4));
    float4 sum = *reinterpret_cast<const float4*>(sums + to * KEYS_O_STRIDE + d);
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const float4 part = *reinterpret_cast<const float4*>(sums + (w * KEYS_BM + to) * KEYS_O_STRIDE + d);
      sum.x += part.x;
      sum.y += part.y;
      sum.z += part.z;
      sum.w += part.w;
    }
    const float inv = inverse[to];
    const float o[4] = {sum.x * inv, sum.y * inv, sum.z * inv, sum.w * inv};
    uint32_t half[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) half[e] = __builtin_bit_cast(uint16_t, static_cast<bf16_t>(o[e]));
    *reinterpret_cast<uint2*>(out + (static_cast<int64_t>(token0 + to) * heads + head) * D + d) =
        uint2{half[0] | (half[1] << 16), half[2] | (half[3] << 16)};
  }
}

// Whether it takes such pages: their bytes are counted in 32 bits, and a lane's place in a head's part of one.
extern "C" int distie_attention_prefill_keys_fits(int kv_heads, int block_size) {
  return kv_heads >= 1 && block_size >= 16 && block_size % 16 == 0 && block_size <= 65536 &&
         2 * static_cast<int64_t>(kv_heads) * block_size * D <= 0xffffffffll;
}

// As distie_attention_prefill_bf16, with nothing between its parts. waves (of a workgroup): 2, 4 or 8.
extern "C" int distie_attention_prefill_keys(const void* qkv, int64_t q_stride, const void* k_cache, const void* v_cache,
                                             const int32_t* positions, const int32_t* cu_q, const int32_t* block_table,
                                             int table_width, const int32_t* table_rows, void* out, int tokens, int num_requests,
                                             int heads, int kv_heads, int block_size, float scale, int window, int min_q_len,
                                             const float* sinks, int waves, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (heads < 1 || !distie_attention_prefill_keys_fits(kv_heads, block_size) || heads % kv_heads != 0 || table_width < 1 || num_requests < 1 || min_q_len < 1 || (waves != 2 && waves != 4 && waves != 8) || !(scale > 0.f))
    return DISTIE_BAD_ARGUMENT;
  const int64_t tiles = (static_cast<int64_t>(tokens) + KEYS_BM - 1) / KEYS_BM + num_requests;     // an upper bound; spare blocks leave at once
  if (tiles > 65535) return DISTIE_BAD_ARGUMENT;
  auto run = [&](auto kernel, int bytes) {
    kernel<<<dim3(heads, static_cast<unsigned>(tiles)), DISTIE_WAVE * waves, bytes, stream>>>(
        static_cast<const bf16_t*>(qkv), q_stride, static_cast<const bf16_t*>(k_cache), static_cast<const bf16_t*>(v_cache),
        positions, cu_q, block_table, table_width, table_rows, static_cast<bf16_t*>(out), num_requests, heads, kv_heads,
        block_size, scale, window, min_q_len, sinks);
    return launch_status();
  };
  return waves == 8 ? run(attn_prefill_keys_kernel<8>, prefill_keys_lds<8>())
                    : waves == 4 ? run(attn_prefill_keys_kernel<4>, prefill_keys_lds<4>())
                                 : run(attn_prefill_keys_kernel<2>, prefill_keys_lds<2>());
}
#else
extern "C" int distie_attention_prefill_keys_fits(int, int) { return 0; }
extern "C" int distie_attention_prefill_keys(const void*, int64_t, const void*, const void*, const int32_t*, const int32_t*,
                                             const int32_t*, int, const int32_t*, void*, int, int, int, int, int, float, int, int,
                                             const float*, int, hipStream_t) {
  return DISTIE_BAD_ARGUMENT;
}
#endif

// ===================================================================================================
//  * attn_prefill_f32: the tiled kernel in float32, for head sizes that are multiples of 32 up to 128. The same
//    walk as attn_prefill (a workgroup of four waves owns 128 new tokens of one head, 32 query columns a wave,
//    K and V^T tiles of 64 keys through LDS, the keys cut into parts that are merged) on the float32 products
//    v_mfma_f32_32x32x2_f32: float32 operands, products and sums, no reduced precision anywhere. Such a product
//    sums over two values, one from each half of the wave; four of them in a row take a lane's 16 bytes of a K or
//    V^T row, so the head dimension (first product) and the keys (second product) are summed in the order in
//    which the lanes hold them: d = 8 g + 4 h + e and key = 8 i + 4 h + j for step e or j of group g or i.
//    The weights stay where the scores were (the accumulators' layout is the B operand's), in float32.
// ===================================================================================================
#if (DISTIE_HEAD_DIM % 32 == 0) && (DISTIE_HEAD_DIM <= 128)
constexpr int PF32_K_STRIDE = D + 4;                    // floats: rows of an odd number of 16-byte pieces
constexpr int PF32_V_STRIDE = PF_BN + 4;
constexpr int PF32_CHUNKS = 4 * D;                      // 16-byte pieces of 16 keys of K ([16, D]), and of V^T ([D, 16])
constexpr int PF32_PASSES = PF32_CHUNKS / DISTIE_WAVE;  // pieces a lane carries per block
constexpr int PF32_AHEAD = 2;                           // reads from LDS ahead of the products (four products a read)

__global__ __launch_bounds__(PF_THREADS, 1) void attn_prefill_f32_kernel(
    const float* __restrict__ qkv, int64_t q_stride, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int32_t* __restrict__ positions, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ table_rows, float* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int tokens, int num_requests, int heads, int kv_heads,
    int block_size, float scale, int window, int min_q_len, const float* __restrict__ sinks) {
  __shared__ __attribute__((aligned(16))) float k_lds[PF_BN * PF32_K_STRIDE];
  __shared__ __attribute__((aligned(16))) float v_lds[D * PF32_V_STRIDE];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / DISTIE_WAVE);
  const int lane = tid % DISTIE_WAVE;
  const int c = lane % 32;
  const int h = lane / 32;
  const int group = heads / kv_heads;
  const float scale_log2 = scale * 1.4426950408889634f;

  // ---- which tokens (as in attn_prefill)
  int tile = gridDim.y - 1 - blockIdx.y;
  int request = 0, begin = 0, end = 0;
  for (; request < num_requests; ++request) {
    begin = cu_q[request];
    end = cu_q[request + 1];
    if (end - begin < min_q_len) continue;
    const int tiles = (end - begin + PF_BM - 1) / PF_BM;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (request >= num_requests) return;
  const int head = blockIdx.x;
  const int kh = head / group;
  const int token0 = begin + tile * PF_BM;
  const int columns = min(PF_BM, end - token0);
  const int pos0 = positions[token0];
  const int key_begin = first_visible(pos0, window);
  const int key_end = pos0 + columns - 1;
  const int32_t* table = block_table + static_cast<int64_t>(table_rows != nullptr ? table_rows[request] : request) * table_width;

  const int wave_col0 = wave * PF_WAVE_COLS;
  const int wave_cols = max(0, min(PF_WAVE_COLS, columns - wave_col0));
  const int wave_last = pos0 + wave_col0 + wave_cols - 1;
  const int wave_first = first_visible(pos0 + wave_col0, window);
  const int wave_open = first_visible(max(wave_last, 0), window);      // from here on every column of the wave sees (up to its own position)
  const int col = min(wave_col0 + c, columns - 1);
  const int col_last = pos0 + col;
  const int col_first = first_visible(col_last, window);
  float4 q_reg[D / 8];                                    // of the lane's column: d = 8 g + 4 h + (0..3)
  {
    const float* q = qkv + (token0 + col) * q_stride + static_cast<int64_t>(head) * D;
#pragma unroll
    for (int g = 0; g < D / 8; ++g) q_reg[g] = *reinterpret_cast<const float4*>(q + 8 * g + 4 * h);
  }
  floatx16 o_acc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) o_acc[db][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // ---- staging: wave w brings block w of the tile (keys k0 + 16 w .. + 15)
  uint4 k_stage[PF32_PASSES], v_stage[PF32_PASSES];
  const int block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  auto block_live = [&](int key) { return key <= key_end && key + 15 >= key_begin; };
  auto lookup = [&](int k0) {
    const int key = k0 + 16 * wave;
    const int slot = block_shift >= 0 ? key >> block_shift : key / block_size;
    return table[min(slot, table_width - 1)];
  };
  auto fetch = [&](int k0, int page_of_block) {
    const int key = k0 + 16 * wave;
    const bool live = block_live(key);
    const int offset = live ? (block_shift >= 0 ? key & (block_size - 1) : key % block_size) : 0;
    const int64_t base = live ? (static_cast<int64_t>(page_of_block) * kv_heads + kh) * block_size * D : 0;
    const float* k_block = k_cache + base + static_cast<int64_t>(offset) * D;
    const float* v_block = v_cache + base + offset;
#pragma unroll
    for (int p = 0; p < PF32_PASSES; ++p) {
      const int j = lane + p * DISTIE_WAVE;
      k_stage[p] = *reinterpret_cast<const uint4*>(k_block + 4 * j);
      v_stage[p] = *reinterpret_cast<const uint4*>(v_block + static_cast<int64_t>(j / 4) * block_size + 4 * (j % 4));
    }
  };
  int k_slot[PF32_PASSES], v_slot[PF32_PASSES];
#pragma unroll
  for (int p = 0; p < PF32_PASSES; ++p) {
    const int j = lane + p * DISTIE_WAVE;
    k_slot[p] = (16 * wave + j / (D / 4)) * PF32_K_STRIDE + 4 * (j % (D / 4));
    v_slot[p] = (j / 4) * PF32_V_STRIDE + 16 * wave + 4 * (j % 4);
  }
  // Slots after the last key of this workgroup were not written by this request, and blocks outside the keys
  // of this workgroup were not read: cleared (a weight of zero times NaN would still be NaN).
  auto stash = [&](int k0) {
    const int key = k0 + 16 * wave;
    const bool live = block_live(key);
    if (live && key + 15 <= key_end) {
#pragma unroll
      for (int p = 0; p < PF32_PASSES; ++p) {
        *reinterpret_cast<uint4*>(k_lds + k_slot[p]) = k_stage[p];
        *reinterpret_cast<uint4*>(v_lds + v_slot[p]) = v_stage[p];
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < PF32_PASSES; ++p) {
      const int j = lane + p * DISTIE_WAVE;
      *reinterpret_cast<uint4*>(k_lds + k_slot[p]) = live ? k_stage[p] : uint4{0u, 0u, 0u, 0u};
      const int written = live ? key_end - (key + 4 * (j % 4)) + 1 : 0;        // of this piece's four keys
      *reinterpret_cast<uint4*>(v_lds + v_slot[p]) =
          uint4{written >= 1 ? v_stage[p].x : 0u, written >= 2 ? v_stage[p].y : 0u, written >= 3 ? v_stage[p].z : 0u,
                written >= 4 ? v_stage[p].w : 0u};
    }
  };

  auto compute = [&](int k0) {
    if (wave_cols <= 0 || k0 > wave_last || k0 + PF_BN - 1 < wave_first) return;
    // ---- scores: 64 keys x the wave's 32 columns, as two blocks of 32 keys
    floatx16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[kb][e] = 0.f;
    {
      float4 a[D / 4];
#pragma unroll
      for (int i = 0; i < D / 4; ++i)
        a[i] = *reinterpret_cast<const float4*>(k_lds + (32 * (i % 2) + c) * PF32_K_STRIDE + 8 * (i / 2) + 4 * h);
#pragma unroll
      for (int i = 0; i < D / 4; ++i) {
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].x, q_reg[i / 2].x, s[i % 2], 0, 0, 0);
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].y, q_reg[i / 2].y, s[i % 2], 0, 0, 0);
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].z, q_reg[i / 2].z, s[i % 2], 0, 0, 0);
        s[i % 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].w, q_reg[i / 2].w, s[i % 2], 0, 0, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, PF32_AHEAD, 0);
#pragma unroll
      for (int i = 0; i < D / 4 - PF32_AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * PF32_AHEAD, 0);
    }
    const bool tile_open = k0 + PF_BN - 1 <= pos0 + wave_col0 &&
                           k0 >= wave_open;
    if (!tile_open) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = k0 + 32 * kb + 8 * (e / 4) + 4 * h + e % 4;
          if (key < col_first || key > col_last) s[kb][e] = -INFINITY;
        }
    }
    // the column's reference follows its largest score when that has outgrown it (see attn_prefill)
    float top = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) top = fmaxf(top, s[kb][e]);
    top = lanes_max<32>(top);
    const float best = top * scale_log2;
    if (__any(best > m_run + PF_GROW)) {
      const float m_new = fmaxf(m_run, best);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o_acc[db][e] *= alpha;
    }
    const float from = m_run == -INFINITY ? 0.f : -m_run;
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[kb][e] = fast_exp2(fmaf(s[kb][e], scale_log2, from));
        sum += s[kb][e];
      }
    l_run += sum;
    // ---- O^T += V^T . P^T: eight groups of four keys for each block of 32 output rows
    {
      constexpr int reads = 8 * (D / 32);
      float4 vt[reads];
#pragma unroll
      for (int i = 0; i < reads; ++i) {
        const int db = i % (D / 32), group_of_keys = i / (D / 32);        // group: kb = / 4, i = % 4
        vt[i] = *reinterpret_cast<const float4*>(v_lds + (32 * db + c) * PF32_V_STRIDE + 8 * group_of_keys + 4 * h);
      }
#pragma unroll
      for (int i = 0; i < reads; ++i) {
        const int db = i % (D / 32), kb = (i / (D / 32)) / 4, e = 4 * ((i / (D / 32)) % 4);
        o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[i].x, s[kb][e], o_acc[db], 0, 0, 0);
        o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[i].y, s[kb][e + 1], o_acc[db], 0, 0, 0);
        o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[i].z, s[kb][e + 2], o_acc[db], 0, 0, 0);
        o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[i].w, s[kb][e + 3], o_acc[db], 0, 0, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, PF32_AHEAD, 1);
#pragma unroll
      for (int i = 0; i < reads - PF32_AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * PF32_AHEAD, 1);
    }
  };

  const int all_tile0 = key_begin / PF_BN * PF_BN;
  const int all_tiles = (key_end - all_tile0) / PF_BN + 1;
  const int per_split = (all_tiles + gridDim.z - 1) / gridDim.z;
  const int tile0 = all_tile0 + static_cast<int>(blockIdx.z) * per_split * PF_BN;
  const int loop_end = min(key_end, tile0 + per_split * PF_BN - 1);
  fetch(tile0, lookup(tile0));
  int page_ahead = lookup(tile0 + PF_BN);
  for (int k0 = tile0; k0 <= loop_end; k0 += PF_BN) {
    __syncthreads();                       // every wave is done with the tile in LDS
    stash(k0);
    __syncthreads();
    fetch(k0 + PF_BN, page_ahead);
    page_ahead = lookup(k0 + 2 * PF_BN);
    compute(k0);
  }
  // ---- write: the lane holds, of its column, output rows 32 db + 8 i + 4 h + (0..3)
  l_run = lanes_sum<32>(l_run);
  if (wave_col0 + c >= columns) return;
  const int64_t row = static_cast<int64_t>(token0 + wave_col0 + c) * heads + head;
  const bool whole = gridDim.z == 1;
  const int64_t at = whole ? row : static_cast<int64_t>(blockIdx.z) * tokens * heads + row;
  float* o = (whole ? out : part_o) + at * D;
  // (a part without a key for this column leaves l = 0: not read)
  const float factor = whole ? sink_factor(m_run, l_run, sinks != nullptr ? sinks[head] * 1.4426950408889634f : -INFINITY) : 1.f;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<float4*>(o + 32 * db + 8 * i + 4 * h) =
          float4{o_acc[db][4 * i] * factor, o_acc[db][4 * i + 1] * factor, o_acc[db][4 * i + 2] * factor, o_acc[db][4 * i + 3] * factor};
  if (!whole && h == 0) {
    part_ml[2 * at] = m_run;
    part_ml[2 * at + 1] = l_run;
  }
}
#endif

extern "C" int distie_attention_prefill_f32_fits() { return (D % 32 == 0 && D <= 128) ? 1 : 0; }

// As distie_attention_prefill_bf16, for float32 queries and a float32 cache; head sizes for which
// distie_attention_prefill_f32_fits() says 1.
extern "C" int distie_attention_prefill_f32(const void* qkv, int64_t q_stride, const void* k_cache, const void* v_cache,
                                            const int32_t* positions, const int32_t* cu_q, const int32_t* block_table,
                                            int table_width, const int32_t* table_rows, void* out, int tokens, int num_requests, int heads,
                                            int kv_heads, int block_size, float scale, int window, int min_q_len,
                                            const int32_t* token_request, float* part_o, float* part_ml,
                                            int splits, const float* sinks, hipStream_t stream) {
#if (DISTIE_HEAD_DIM % 32 == 0) && (DISTIE_HEAD_DIM <= 128)
  if (tokens <= 0) return 0;
  if (heads < 1 || kv_heads < 1 || heads % kv_heads != 0 || block_size % 16 != 0 || table_width < 1 ||
      num_requests < 1 || heads > 65535 || min_q_len < 1 || splits < 1 || splits > PF_MAX_SPLITS || !(scale > 0.f) ||
      q_stride % 4 != 0 ||
      (splits > 1 && (part_o == nullptr || part_ml == nullptr || token_request == nullptr)))
    return DISTIE_BAD_ARGUMENT;
  const int tiles = (tokens + PF_BM - 1) / PF_BM + num_requests;
  if (tiles > 65535) return DISTIE_BAD_ARGUMENT;
  attn_prefill_f32_kernel<<<dim3(heads, tiles, splits), PF_THREADS, 0, stream>>>(
      static_cast<const float*>(qkv), q_stride, static_cast<const float*>(k_cache), static_cast<const float*>(v_cache),
      positions, cu_q, block_table, table_width, table_rows, static_cast<float*>(out), part_o, part_ml, tokens, num_requests,
      heads, kv_heads, block_size, scale, window, min_q_len, sinks);
  int status = launch_status();
  if (status != 0 || splits == 1) return status;
  launch_merge(part_o, part_ml, token_request, cu_q, static_cast<float*>(out), tokens, heads, min_q_len, splits, sinks, stream);
  return launch_status();
#else
  return DISTIE_BAD_ARGUMENT;
#endif
}

#else   // a head size that is no multiple of 16: the wave-per-token kernel is all there is

extern "C" int distie_attention_decode_columns() { return 0; }

extern "C" int distie_attention_decode_bf16(const void*, int64_t, const void*, const void*, const int32_t*, const int32_t*,
                                            const int32_t*, int, const int32_t*, void*, void*, void*, int, int, int, int, float, int, int,
                                            int, int, const int32_t*, const float*, int, hipStream_t) {
  return DISTIE_BAD_ARGUMENT;
}

extern "C" int distie_attention_decode_together(int, int, int) { return 1; }

extern "C" int distie_attention_decode_run_len(const int32_t*, int, int, int, int32_t*, hipStream_t) { return DISTIE_BAD_ARGUMENT; }

extern "C" int distie_attention_prefill_bf16(const void*, int64_t, const void*, const void*, const int32_t*, const int32_t*,
                                             const int32_t*, int, const int32_t*, void*, int, int, int, int, int, float, int, int,
                                             const int32_t*, void*, void*, int, const float*, hipStream_t) {
  return DISTIE_BAD_ARGUMENT;
}

extern "C" int distie_attention_prefill_keys_fits(int, int) { return 0; }

extern "C" int distie_attention_prefill_keys(const void*, int64_t, const void*, const void*, const int32_t*, const int32_t*,
                                             const int32_t*, int, const int32_t*, void*, int, int, int, int, int, float, int, int,
                                             const float*, int, hipStream_t) {
  return DISTIE_BAD_ARGUMENT;
}

extern "C" int distie_attention_prefill_f32_fits() { return 0; }

extern "C" int distie_attention_prefill_f32(const void*, int64_t, const void*, const void*, const int32_t*, const int32_t*,
                                            const int32_t*, int, const int32_t*, void*, int, int, int, int, int, float, int, int,
                                            const int32_t*, void*, void*, int, const float*, hipStream_t) {
  return DISTIE_BAD_ARGUMENT;
}

#endif
