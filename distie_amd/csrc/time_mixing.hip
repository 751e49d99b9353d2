// Time mixing with a token shift and a state whose decay is computed from the token, with a bonus for the current token.
//
// A step is a flattened batch: token t belongs to request token_request[t], whose new tokens are rows
// cu_q[b] .. cu_q[b+1]-1 and whose states are rows state_slots[b] of the state tensors. Decays with their
// exponentials, the state and every sum into it, head norms and gates are float32 in either precision.
#include "common.h"
#include "vector_values.h"

namespace {

constexpr int SHIFT_MAX_MIXES = 8;

// out[k][t] = x_t + (x_(t-1) - x_t) * mu[k] for every mix k; the row before a request's first row of the step is its
// state row. The thread that reads a state value is the one that replaces it by the request's last row of the step.
template <int V, typename X>
__global__ void token_shift_kernel(const X* __restrict__ x, const float* __restrict__ mu, int mixes, float* __restrict__ state,
                                   X* __restrict__ out, const int32_t* __restrict__ cu_q,
                                   const int32_t* __restrict__ token_request, const int32_t* __restrict__ state_slots, int C,
                                   int64_t T) {
  const int64_t t = blockIdx.x;
  const int c = V * static_cast<int>(blockIdx.y * blockDim.x + threadIdx.x);
  if (c >= C) return;
  const int b = token_request != nullptr ? token_request[t] : static_cast<int>(t);     // null: a row a request
  const int64_t first = token_request != nullptr ? cu_q[b] : t;
  float h[V], before[V];
  load_values<V>(x + t * C + c, h);
  if (t > first) {
    load_values<V>(x + (t - 1) * C + c, before);
  } else {
    float* own = state + static_cast<int64_t>(state_slots[b]) * C + c;
    const int64_t last = token_request != nullptr ? cu_q[b + 1] - 1 : t;
    float keep[V];
    load_values<V>(own, before);
    load_values<V>(x + last * C + c, keep);
    store_values<V>(own, keep);
  }
#pragma unroll
  for (int k = 0; k < V; ++k) before[k] -= h[k];
  for (int m = 0; m < mixes; ++m) {
    float w[V], v[V];
    load_values<V>(mu + static_cast<int64_t>(m) * C + c, w);
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = h[k] + before[k] * w[k];
    store_values<V>(out + (m * T + t) * C + c, v);
  }
}

// ---------------------------------------------------------------------------------------------------
// Row after row. A block owns one head of one request: thread (part, e) keeps rows d = part, part + PARTS, ... of column e
// of the state in registers. Per token: the decay of every key channel from `low` (tanh, the second projection, both
// exponentials; `z` instead of `low` where the projection was made before), then
//   o[e] = sum_d r[d] (S[d][e] + u[d] k[d] v[e]);   S[d][e] = w[d] S[d][e] + k[d] v[e]
// the PARTS partial sums of a column meet in LDS, the head's norm is taken over its D columns, times its weight and
// silu(gate). The next token's values are asked for before this token's are used.
template <typename X, typename L, typename O, int COLS, int PARTS, int ROWS>
__global__ void __launch_bounds__(COLS * PARTS)
wkv_scan_kernel(const X* __restrict__ r_in, const X* __restrict__ k_in, const X* __restrict__ v_in,
                const X* __restrict__ gates, int64_t ld, const L* __restrict__ low, int64_t ld_low, int rank,
                const float* __restrict__ up, const float* __restrict__ up_bias, const float* __restrict__ bonus,
                float* __restrict__ state, const float* __restrict__ norm_weight, float eps, O* __restrict__ out,
                const int32_t* __restrict__ cu_q, const int32_t* __restrict__ state_slots, int H, int D) {
  extern __shared__ float low_s[];                         // [rank]
  __shared__ float r_s[PARTS * ROWS], k_s[PARTS * ROWS], w_s[PARTS * ROWS], u_s[PARTS * ROWS];
  __shared__ float partial[PARTS][COLS];
  __shared__ float squares[COLS / 64];
  constexpr int THREADS = COLS * PARTS;
  constexpr int SUB = THREADS / (PARTS * ROWS);            // threads that share a channel's decay (4 at least, a power of two)
  const int b = blockIdx.x, head = blockIdx.y;
  const int e = threadIdx.x % COLS, part = threadIdx.x / COLS;
  const int first = cu_q != nullptr ? cu_q[b] : b, last = cu_q != nullptr ? cu_q[b + 1] : b + 1;     // null: a row a request
  if (first >= last) return;
  float* own = state + (static_cast<int64_t>(state_slots[b]) * H + head) * D * D;
  float s[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int d = part + i * PARTS;
    s[i] = (d < D && e < D) ? own[static_cast<int64_t>(d) * D + e] : 0.f;
  }
  const int d_own = threadIdx.x;                           // the channel whose r and k this thread fetches
  const int channel = threadIdx.x / SUB, sub = threadIdx.x % SUB;      // the channel whose decay it helps to make
  const float* up_row = up + static_cast<int64_t>(head * D + min(channel, D - 1)) * rank;
  const float z0 = up_bias[head * D + min(channel, D - 1)];
  constexpr int UP_HELD = 16;                              // of the channel's row, kept for all tokens
  float up_held[UP_HELD];
#pragma unroll
  for (int i = 0; i < UP_HELD; ++i) up_held[i] = sub + i * SUB < rank ? up_row[sub + i * SUB] : 0.f;
  if (d_own < D) u_s[d_own] = bonus[head * D + d_own];
  const float weight = e < D ? norm_weight[head * D + e] : 0.f;
  float nr = 0.f, nk = 0.f, nv = 0.f, ng = 0.f, nl = 0.f;
  auto fetch = [&](int t) {
    const int64_t row = static_cast<int64_t>(t) * ld + head * D;
    if (d_own < D) nr = to_float(r_in[row + d_own]), nk = to_float(k_in[row + d_own]);
    if (e < D) nv = to_float(v_in[row + e]), ng = to_float(gates[row + e]);
    if (threadIdx.x < rank) nl = to_float(low[static_cast<int64_t>(t) * ld_low + threadIdx.x]);
  };
  fetch(first);
  for (int t = first; t < last; ++t) {
    if (threadIdx.x < rank) low_s[threadIdx.x] = tanhf(nl);
    for (int i = threadIdx.x + THREADS; i < rank; i += THREADS)
      low_s[i] = tanhf(to_float(low[static_cast<int64_t>(t) * ld_low + i]));
    if (d_own < D) r_s[d_own] = nr, k_s[d_own] = nk;
    const float v = nv, g = ng;
    if (t + 1 < last) fetch(t + 1);
    __syncthreads();
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < UP_HELD; ++i) z += up_held[i] * (sub + i * SUB < rank ? low_s[sub + i * SUB] : 0.f);
    for (int i = sub + UP_HELD * SUB; i < rank; i += SUB) z += up_row[i] * low_s[i];
#pragma unroll
    for (int o = SUB / 2; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
    if (sub == 0 && channel < D) w_s[channel] = expf(-expf(z + z0));
    __syncthreads();
    float o = 0.f;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int d = part + i * PARTS;
      if (d < D) {
        const float kv = k_s[d] * v;
        o += r_s[d] * (s[i] + u_s[d] * kv);
        s[i] = w_s[d] * s[i] + kv;
      }
    }
    partial[part][e] = o;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int p = 0; p < PARTS; ++p) total += partial[p][e];
    float sq = wave_sum(e < D ? total * total : 0.f);
    if constexpr (COLS > 64) {
      if (part == 0 && e % 64 == 0) squares[e / 64] = sq;
      __syncthreads();
      sq = 0.f;
#pragma unroll
      for (int i = 0; i < COLS / 64; ++i) sq += squares[i];
    }
    if (part == 0 && e < D)
      out[(static_cast<int64_t>(t) * H + head) * D + e] =
          from_float<O>(total / sqrtf(sq / D + eps) * weight * (g / (1.f + expf(-g))));
    // (the next token's values go to other places of LDS than what is read behind the last barrier, but for the
    // partial sums and the squares, which two barriers stand in front of)
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int d = part + i * PARTS;
    if (d < D && e < D) own[static_cast<int64_t>(d) * D + e] = s[i];
  }
}

// ---------------------------------------------------------------------------------------------------
// The same recurrence over portions of prompts, in chunks of 64 rows that run side by side. With S the state in front of
// a chunk and c_i the sum of ln w over its rows up to and with i:
//   sums:     P[d][e] = sum_j exp(c_L[d] - c_j[d]) k_j[d] v_j[e],   G[d] = exp(c_L[d])            (each chunk alone)
//   states:   S_next = diag(G) S + P, chunk after chunk; the state in front of a chunk takes P's place
//   outputs:  o_i[e] = sum_d r_i[d] exp(c_(i-1)[d]) S[d][e] + sum_(j < i) (sum_d r_i[d] k_j[d] exp(c_(i-1)[d] - c_j[d])) v_j[e]
//                      + (sum_d r_i[d] u[d] k_i[d]) v_i[e]
// and behind them head norm, weight and gate. Everything is float32, the tiles' products on v_mfma_f32_16x16x4_f32.
//
// A chunk is four runs of 16 rows, a wave each. A wave's lane (i = lane % 16, g = lane / 16) owns row i of the run and the
// channels DL g .. DL g + DL - 1 (DL = DP / 4) of r, k and ln w: the matrix cores' operand with the summed index in an order
// of our own. Sums of ln w run over the rows of one run only, by row shifts between the lanes; what lies between two runs
// enters as a product of the runs' total factors. So every exponent is <= 0, no quotient of decays is formed, and differences
// are taken over 16 rows at most. The scores between different runs are products of the matrix cores, taken transposed:
// their result lies as the next product's operand. Those within a run need an exponential of their own for every pair and
// channel: row j of k and ln w goes to all lanes of its group by a row broadcast.
constexpr int WK_ROWS = 64;
constexpr float LOG2E = 1.4426950408889634f;

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

template <int CTRL>
__device__ __forceinline__ float row_move(float x) {          // a DPP move within rows of 16 lanes; 0 where nothing comes in
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float row_shift(float x) { return row_move<0x110 + N>(x); }       // from the lane N below
template <int N>
__device__ __forceinline__ float row_lane(float x) { return row_move<0x150 + N>(x); }        // lane N of the row, to all

__device__ __forceinline__ float groups_sum(float v) {        // over the four lanes that own a row
  return lanes_sum<32>(lanes_sum<16>(v));
}

// a lane's channels of one row of a head (`row` points at the head's first column); zeros for a row that is not there
template <int DP, typename X>
__device__ __forceinline__ void load_channels(const X* __restrict__ row, int D, int g, bool there, float out[DP / 4]) {
  constexpr int DL = DP / 4;
#pragma unroll
  for (int s = 0; s < DL; ++s) out[s] = 0.f;
  if (!there) return;
#pragma unroll
  for (int s = 0; s < DL; ++s)
    if (DL * g + s < D) out[s] = to_float(row[DL * g + s]);
}

// Four neighbouring values as they lie in memory: asked for here, turned into float32 where they are needed.
template <typename X> struct Four;
template <> struct Four<float> {
  float4 raw;
  __device__ __forceinline__ void load(const float* p) { raw = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void values(bool there, float v[4]) const {
    v[0] = there ? raw.x : 0.f, v[1] = there ? raw.y : 0.f, v[2] = there ? raw.z : 0.f, v[3] = there ? raw.w : 0.f;
  }
};
template <> struct Four<bf16_t> {
  uint2 raw;
  __device__ __forceinline__ void load(const bf16_t* p) { raw = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ void values(bool there, float v[4]) const {
    const uint32_t a = there ? raw.x : 0u, b = there ? raw.y : 0u;
    v[0] = __uint_as_float(a << 16), v[1] = __uint_as_float(a & 0xffff0000u);
    v[2] = __uint_as_float(b << 16), v[3] = __uint_as_float(b & 0xffff0000u);
  }
};


// `loads_first` behind what a lane needs at the start makes that one trip to memory. (Left to itself, and with a choice at every load between
// whole heads and others, the compiler waited for r, k, ln w, each piece of V and the state one after the other: 2 prompts of 901, 32 heads
// of 64, outputs 42.2 -> 38.2 us, sums 16.3 -> 15.6; four workgroups a compute unit hid the rest.)
// a lane's channels of a row of a whole head, which is there in memory whether it counts or not
template <int DP, typename X>
__device__ __forceinline__ void ask_channels(const X* __restrict__ row, int g, Four<X> (&raw)[DP / 16]) {
#pragma unroll
  for (int s = 0; s < DP / 16; ++s) raw[s].load(row + DP / 4 * g + 4 * s);
}
template <int DP, typename X>
__device__ __forceinline__ void take_channels(const Four<X> (&raw)[DP / 16], bool there, float out[DP / 4]) {
#pragma unroll
  for (int s = 0; s < DP / 16; ++s) raw[s].values(there, out + 4 * s);
}

// log2 of the decays of a lane's channels (c: ln of minus their ln), summed over the rows of the run up to the lane's own
template <int DP>
__device__ __forceinline__ void sum_decays(bool there, float c[DP / 4]) {
#pragma unroll
  for (int s = 0; s < DP / 4; ++s) {
    // (a factor of 2^-160 is zero in float32: smaller ones need no larger exponents, and infinities have no differences)
    c[s] = there ? fmaxf(-LOG2E * expf(c[s]), -160.f) : 0.f;
    c[s] += row_shift<1>(c[s]);
    c[s] += row_shift<2>(c[s]);
    c[s] += row_shift<4>(c[s]);
    c[s] += row_shift<8>(c[s]);
  }
}

// V of a chunk into LDS as float32, rows DP + 4 apart, zeros for what is not there
template <int DP, typename X>
__device__ __forceinline__ void stage_rows(const X* __restrict__ v, int64_t ld, int len, int D, float* __restrict__ to) {
  constexpr int RUNS = DP / 4;
  for (int idx = threadIdx.x; idx < WK_ROWS * RUNS; idx += blockDim.x) {
    const int j = idx / RUNS, e = idx % RUNS * 4;
    float x[4] = {};
    if (j < len) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (e + k < D) x[k] = to_float(v[j * ld + e + k]);
    }
    store_values<4>(to + j * (DP + 4) + e, x);
  }
}

// The same of whole heads, in two halves: a thread's pieces, and their places in LDS.
template <int DP, typename X>
__device__ __forceinline__ void ask_rows(const X* __restrict__ v, int64_t ld, int len, Four<X> (&raw)[DP / 16]) {
#pragma unroll
  for (int p = 0; p < DP / 16; ++p) {
    const int idx = threadIdx.x + 256 * p;
    raw[p].load(v + min(idx / (DP / 4), len - 1) * ld + idx % (DP / 4) * 4);
  }
}
template <int DP, typename X>
__device__ __forceinline__ void put_rows(const Four<X> (&raw)[DP / 16], int len, float* __restrict__ to) {
#pragma unroll
  for (int p = 0; p < DP / 16; ++p) {
    const int idx = threadIdx.x + 256 * p, j = idx / (DP / 4);
    float x[4];
    raw[p].values(j < len, x);
    store_values<4>(to + j * (DP + 4) + idx % (DP / 4) * 4, x);
  }
}

// WHOLE: D is DP, and everything begins where four values may be loaded at once
template <int DP, bool WHOLE, typename X>
__global__ void __launch_bounds__(256)
wkv_chunk_sums_kernel(const X* __restrict__ k_in, const X* __restrict__ v_in, int64_t ld, const float* __restrict__ z,
                      float* __restrict__ scratch, float* __restrict__ totals, const int4* __restrict__ chunks, int H, int D) {
  constexpr int DL = DP / 4, STRIDE = DP + 4;
  __shared__ __attribute__((aligned(16))) float Ks[WK_ROWS * STRIDE];
  __shared__ __attribute__((aligned(16))) float Vs[WK_ROWS * STRIDE];
  __shared__ float factor[4][DP];
  const int head = blockIdx.y;
  const int4 chunk = chunks[blockIdx.x];
  const int64_t row0 = chunk.y;
  const int len = chunk.z;
  const int lane = threadIdx.x % 64, run = threadIdx.x / 64, i = lane % 16, g = lane / 16;
  const int row = 16 * run + i;
  float k[DL], c[DL];
  if constexpr (WHOLE) {
    const int64_t at = row0 + min(row, len - 1);
    Four<X> k4[DP / 16], v4[DP / 16];
    Four<float> z4[DP / 16];
    ask_channels<DP>(z + (at * H + head) * D, g, z4);
    ask_channels<DP>(k_in + at * ld + head * D, g, k4);
    ask_rows<DP>(v_in + row0 * ld + head * D, ld, len, v4);
    loads_first();
    take_channels<DP>(z4, row < len, c);
    take_channels<DP>(k4, row < len, k);
    put_rows<DP>(v4, len, Vs);
  } else {
    load_channels<DP>(k_in + (row0 + row) * ld + head * D, D, g, row < len, k);
    load_channels<DP>(z + ((row0 + row) * H + head) * D, D, g, row < len, c);
    stage_rows<DP>(v_in + row0 * ld + head * D, ld, len, D, Vs);
  }
  sum_decays<DP>(row < len, c);
#pragma unroll
  for (int s = 0; s < DL; ++s) {
    const float total = row_lane<15>(c[s]);
    k[s] *= __builtin_amdgcn_exp2f(total - c[s]);
    if (i == 0) factor[run][DL * g + s] = __builtin_amdgcn_exp2f(total);
  }
  __syncthreads();
  for (int later = run + 1; later < 4; ++later) {
#pragma unroll
    for (int s = 0; s < DL; ++s) k[s] *= factor[later][DL * g + s];
  }
#pragma unroll
  for (int s = 0; s < DL; s += 4) store_values<4>(Ks + row * STRIDE + DL * g + s, k + s);
  if (threadIdx.x < D)
    totals[(static_cast<int64_t>(blockIdx.x) * H + head) * D + threadIdx.x] =
        factor[0][threadIdx.x] * factor[1][threadIdx.x] * factor[2][threadIdx.x] * factor[3][threadIdx.x];
  __syncthreads();
  float* dst = scratch + (static_cast<int64_t>(blockIdx.x) * H + head) * D * D;
  for (int tile = run; tile < DP / 16; tile += 4) {
    floatx4 acc[DP / 16];
#pragma unroll
    for (int e = 0; e < DP / 16; ++e) acc[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int at = (16 * m + 4 * g + s) * STRIDE + i;
        const float a = Ks[at + 16 * tile];
#pragma unroll
        for (int e = 0; e < DP / 16; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Vs[at + 16 * e], acc[e], 0, 0, 0);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * tile + 4 * g + r;
      if (d >= D) continue;
#pragma unroll
      for (int e = 0; e < DP / 16; ++e)
        if (16 * e + i < D) dst[static_cast<int64_t>(d) * D + 16 * e + i] = acc[e][r];
    }
  }
}

__global__ void wkv_chunk_states_kernel(float* __restrict__ scratch, const float* __restrict__ totals,
                                        float* __restrict__ state, const int32_t* __restrict__ request_chunks,
                                        const int32_t* __restrict__ state_slots, int H, int D) {
  const int b = blockIdx.x, head = blockIdx.y;
  const int idx = blockIdx.z * blockDim.x + threadIdx.x;
  if (idx >= D * D) return;
  const int c0 = request_chunks[b], c1 = request_chunks[b + 1];
  if (c0 >= c1) return;
  float* own = state + (static_cast<int64_t>(state_slots[b]) * H + head) * D * D + idx;
  const int64_t stride = static_cast<int64_t>(H) * D * D;
  float* p = scratch + (static_cast<int64_t>(c0) * H + head) * D * D + idx;
  const float* factor = totals + (static_cast<int64_t>(c0) * H + head) * D + idx / D;
  float S = *own;
  for (int c = c0; c < c1; c += 8) {
    // the sums of eight chunks are asked for together; each then gives way to the state in front of its chunk
    float add[8], keep[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int at = min(u, c1 - 1 - c);
      add[u] = p[at * stride];
      keep[u] = factor[static_cast<int64_t>(at) * H * D];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (c + u >= c1) break;
      p[u * stride] = S;
      S = keep[u] * S + add[u];
    }
    p += 8 * stride;
    factor += 8 * static_cast<int64_t>(H) * D;
  }
  *own = S;
}

// the scores of a run's rows against its own row J, for one J after the other: lane (i, g) gets column 4 g + s in `a[s]`
template <int J, int DP>
__device__ __forceinline__ void run_scores(const float r[DP / 4], const float k[DP / 4], const float x[DP / 4],
                                           const float c[DP / 4], int i, int g, float a[4]) {
  if constexpr (J < 15) {
    float sum = 0.f;
#pragma unroll
    for (int s = 0; s < DP / 4; ++s) sum += r[s] * row_lane<J>(k[s]) * __builtin_amdgcn_exp2f(fminf(x[s] - row_lane<J>(c[s]), 0.f));
    sum = groups_sum(sum);
    if (g == J / 4) a[J % 4] = i > J ? sum : 0.f;
    run_scores<J + 1, DP>(r, k, x, c, i, g, a);
  }
}

// LATE (heads of up to 64, more than WK_EARLY_WORKGROUPS workgroups): the state in front of the chunk waits in registers and takes
// the place of Kt in LDS when that has been read, 35 KB instead of 51, and with 128 registers a lane four workgroups fit a compute unit
// instead of three: 960 of them (2 prompts of 901, 32 heads) 50.4 -> 45.9 us, the same bits (with 130 registers and three of them 50.9).
// Workgroups that all fit as they are gain nothing from it and wait for the state at the end instead: 16 of 20 rows 15.3 -> 16.7 us.
// (The whole operation, early / late: 32 heads, 768 workgroups of 30 rows 85.1 / 86.0 us, 832 of them 94.8 / 92.3.)
constexpr int WK_EARLY_WORKGROUPS = 3 * 256;
template <int DP, bool LATE>
constexpr int wk_shared() {
  const int k = WK_ROWS * DP, s = DP * DP;
  return LATE ? (k > s ? k : s) : k + s;
}

template <int DP, bool LATE, bool WHOLE, typename X, typename O>
__global__ void __launch_bounds__(256, LATE ? 4 : 2)
wkv_chunk_outputs_kernel(const X* __restrict__ r_in, const X* __restrict__ k_in, const X* __restrict__ v_in,
                         const X* __restrict__ gates, int64_t ld, const float* __restrict__ z, const float* __restrict__ bonus,
                         const float* __restrict__ scratch, const float* __restrict__ norm_weight, float eps,
                         O* __restrict__ out, const int4* __restrict__ chunks, int H, int D) {
  constexpr int DL = DP / 4, STRIDE = DP + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* Vs = lds;                                  // [64][DP + 4]
  float* Kt = Vs + WK_ROWS * STRIDE;                // [4 runs][DL / 4][64 lanes][4]: k_j exp(the run's decay behind j)
  float* Ss = LATE ? Kt : Kt + WK_ROWS * DP;        // [DP][DP], the columns of row d turned by 16 (d / DL) places
  float* factor = Kt + wk_shared<DP, LATE>();       // [4][DP]: the runs' total factors
  const int head = blockIdx.y;
  const int4 chunk = chunks[blockIdx.x];
  const int64_t row0 = chunk.y;
  const int len = chunk.z;
  const int lane = threadIdx.x % 64, run = threadIdx.x / 64, i = lane % 16, g = lane / 16;
  const int row = 16 * run + i;
  float r[DL], k[DL], c[DL], x[DL];
  const float* src = scratch + (static_cast<int64_t>(blockIdx.x) * H + head) * D * D;
  constexpr int PIECES = (DP * DP / 4 + 255) / 256; // of S, a thread's
  float held[LATE ? PIECES : 1][4];
  auto load_state = [&](int idx, float v[4]) __attribute__((always_inline)) {
    const int d = idx / (DP / 4), e = idx % (DP / 4) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = 0.f;
    if constexpr (WHOLE) {
      load_values<4>(src + static_cast<int64_t>(min(d, DP - 1)) * D + e, v);
    } else if (d < D) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (e + q < D) v[q] = src[static_cast<int64_t>(d) * D + e + q];
    }
  };
  float u[DL];                                      // the bonus
  if constexpr (WHOLE) {
    const int64_t at = row0 + min(row, len - 1);
    Four<X> r4[DP / 16], k4[DP / 16], v4[DP / 16];
    Four<float> z4[DP / 16], u4[DP / 16];
    ask_channels<DP>(z + (at * H + head) * D, g, z4);
    ask_channels<DP>(k_in + at * ld + head * D, g, k4);
    ask_channels<DP>(r_in + at * ld + head * D, g, r4);
    ask_rows<DP>(v_in + row0 * ld + head * D, ld, len, v4);
    ask_channels<DP>(bonus + head * D, g, u4);
    if constexpr (LATE) {
#pragma unroll
      for (int p = 0; p < PIECES; ++p) load_state(threadIdx.x + 256 * p, held[p]);
    }
    loads_first();
    take_channels<DP>(z4, row < len, c);
    take_channels<DP>(k4, row < len, k);
    take_channels<DP>(r4, row < len, r);
    take_channels<DP>(u4, true, u);
    put_rows<DP>(v4, len, Vs);
  } else {
    load_channels<DP>(r_in + (row0 + row) * ld + head * D, D, g, row < len, r);
    load_channels<DP>(k_in + (row0 + row) * ld + head * D, D, g, row < len, k);
    load_channels<DP>(z + ((row0 + row) * H + head) * D, D, g, row < len, c);
    load_channels<DP>(bonus + head * D, D, g, true, u);
    stage_rows<DP>(v_in + row0 * ld + head * D, ld, len, D, Vs);
  }
  sum_decays<DP>(row < len, c);
  auto stage_state = [&](int idx, const float v[4]) __attribute__((always_inline)) {
    const int d = idx / (DP / 4), e = idx % (DP / 4) * 4;
    if (DP * DP / 4 % 256 == 0 || d < DP) store_values<4>(Ss + d * DP + (e + 16 * (d / DL)) % DP, v);
  };
  if constexpr (LATE) {
    if constexpr (!WHOLE) {
#pragma unroll
      for (int p = 0; p < PIECES; ++p) load_state(threadIdx.x + 256 * p, held[p]);
    }
  } else {
    for (int idx = threadIdx.x; idx < DP * DP / 4; idx += 256) {
      float v[4];
      load_state(idx, v);
      stage_state(idx, v);
    }
  }
#pragma unroll
  for (int s = 0; s < DL; s += 4) {
    float kt[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float total = row_lane<15>(c[s + q]);
      kt[q] = k[s + q] * __builtin_amdgcn_exp2f(total - c[s + q]);
      if (i == 0) factor[run * DP + DL * g + s + q] = __builtin_amdgcn_exp2f(total);
    }
    store_values<4>(Kt + ((run * (DL / 4) + s / 4) * 64 + lane) * 4, kt);
  }
  float own = 0.f;
#pragma unroll
  for (int s = 0; s < DL; ++s) {
    x[s] = row_shift<1>(c[s]);
    own += r[s] * u[s] * k[s];                      // (zeros beyond D)
  }
  own = groups_sum(own);
  float a[4] = {};
  run_scores<0, DP>(r, k, x, c, i, g, a);
#pragma unroll
  for (int s = 0; s < 4; ++s)
    if (4 * g + s == i) a[s] = own;
#pragma unroll
  for (int s = 0; s < DL; ++s) r[s] *= __builtin_amdgcn_exp2f(x[s]);
  __syncthreads();
  floatx4 acc[DP / 16];
#pragma unroll
  for (int e = 0; e < DP / 16; ++e) acc[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < DP / 16; ++e)
      acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], Vs[(16 * run + 4 * g + s) * STRIDE + 16 * e + i], acc[e], 0, 0, 0);
  for (int before = run - 1; before >= 0; --before) {
    floatx4 scores = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DL; s += 4) {
      float kt[4];
      load_values<4>(Kt + ((before * (DL / 4) + s / 4) * 64 + lane) * 4, kt);
#pragma unroll
      for (int q = 0; q < 4; ++q) scores = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[q], r[s + q], scores, 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < DP / 16; ++e)
        acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(scores[s], Vs[(16 * before + 4 * g + s) * STRIDE + 16 * e + i], acc[e], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < DL; ++s) r[s] *= factor[before * DP + DL * g + s];
  }
  if constexpr (LATE) {
    __syncthreads();                                // every run has read Kt
#pragma unroll
    for (int p = 0; p < PIECES; ++p) stage_state(threadIdx.x + 256 * p, held[p]);
    __syncthreads();
  }
#pragma unroll
  for (int s = 0; s < DL; ++s)
#pragma unroll
    for (int e = 0; e < DP / 16; ++e)
      acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[s], Ss[(DL * g + s) * DP + (16 * e + i + 16 * g) % DP], acc[e], 0, 0, 0);
  // lane (i, g) now holds rows 4 g .. 4 g + 3 of the run, column i of every 16; their gates and weights, together
  X gate_of[4][DP / 16];
  float weight[DP / 16];
#pragma unroll
  for (int e = 0; e < DP / 16; ++e) weight[e] = norm_weight[head * D + min(16 * e + i, D - 1)];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < DP / 16; ++e)
      gate_of[q][e] = gates[(row0 + min(16 * run + 4 * g + q, len - 1)) * ld + head * D + min(16 * e + i, D - 1)];
  loads_first();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float sq = 0.f;
#pragma unroll
    for (int e = 0; e < DP / 16; ++e) sq += acc[e][q] * acc[e][q];
    sq = lanes_sum<1>(lanes_sum<2>(lanes_sum<4>(lanes_sum<8>(sq))));
    const float scale = 1.f / sqrtf(sq / D + eps);
    const int at = 16 * run + 4 * g + q;
    const int64_t t = row0 + at;
#pragma unroll
    for (int e = 0; e < DP / 16; ++e) {
      const int col = 16 * e + i;
      const float gate = to_float(gate_of[q][e]);
      const float value = acc[e][q] * scale * weight[e] * (gate / (1.f + expf(-gate)));
      if (at < len && col < D) out[(t * H + head) * D + col] = from_float<O>(value);
    }
  }
}

__global__ void tanh_f32_kernel(const float* __restrict__ in, int64_t ld, float* __restrict__ out, int N, int64_t T) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= T * N) return;
  out[i] = tanhf(in[i / N * ld + i % N]);
}

}  // namespace

extern "C" int distie_token_shift(const void* x, int dtype, const float* mu, int mixes, float* state, void* out,
                                  const int32_t* cu_q, const int32_t* token_request, const int32_t* state_slots, int T, int C,
                                  hipStream_t stream) {
  if (T <= 0) return 0;
  if (C < 1 || mixes < 1 || mixes > SHIFT_MAX_MIXES) return DISTIE_BAD_ARGUMENT;
  const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool wide = C % 8 == 0 && aligned(x) && aligned(mu) && aligned(state) && aligned(out);
  const int runs = wide ? C / 8 : C;
  const int threads = runs >= 256 ? 256 : (runs > 64 ? 128 : 64);
  const dim3 grid(T, (runs + threads - 1) / threads);
  if (wide) {
    DISTIE_DISPATCH(dtype, X, (token_shift_kernel<8, X><<<grid, threads, 0, stream>>>(
        static_cast<const X*>(x), mu, mixes, state, static_cast<X*>(out), cu_q, token_request, state_slots, C, T)));
  } else {
    DISTIE_DISPATCH(dtype, X, (token_shift_kernel<1, X><<<grid, threads, 0, stream>>>(
        static_cast<const X*>(x), mu, mixes, state, static_cast<X*>(out), cu_q, token_request, state_slots, C, T)));
  }
  return launch_status();
}

extern "C" int distie_wkv_scan_max_dim() { return 256; }
extern "C" int distie_wkv_scan_max_rank() { return 8192; }

// r, k, v, gates: [T, H * D] of `dtype` with rows `ld` apart; low: [T, rank] of `low_dtype`, rows `ld_low` apart
extern "C" int distie_wkv_scan(const void* r, const void* k, const void* v, const void* gates, int dtype, int64_t ld,
                               const void* low, int low_dtype, int64_t ld_low, int rank, const float* up,
                               const float* up_bias, const float* bonus, float* state, const float* norm_weight, float eps,
                               void* out, int out_dtype, const int32_t* cu_q, const int32_t* state_slots, int B, int H,
                               int D, hipStream_t stream) {
  if (B <= 0) return 0;
  if (H < 1 || D < 1 || D > 256 || rank < 1 || rank > 8192 || ld < static_cast<int64_t>(H) * D || ld_low < rank || !(eps >= 0.f))
    return DISTIE_BAD_ARGUMENT;
  const dim3 grid(B, H);
  const size_t lds = static_cast<size_t>(rank) * sizeof(float);
#define DISTIE_WKV_SCAN(COLS, PARTS, ROWS)                                                                               \
  DISTIE_DISPATCH(dtype, X, DISTIE_DISPATCH(low_dtype, L, DISTIE_DISPATCH(out_dtype, O, (                                \
      wkv_scan_kernel<X, L, O, COLS, PARTS, ROWS><<<grid, COLS * PARTS, lds, stream>>>(                                  \
          static_cast<const X*>(r), static_cast<const X*>(k), static_cast<const X*>(v), static_cast<const X*>(gates),    \
          ld, static_cast<const L*>(low), ld_low, rank, up, up_bias, bonus, state, norm_weight, eps,                     \
          static_cast<O*>(out), cu_q, state_slots, H, D)))))
  if (D <= 32) {
    DISTIE_WKV_SCAN(64, 4, 8);
  } else if (D <= 64) {
    DISTIE_WKV_SCAN(64, 4, 16);
  } else if (D <= 128) {
    DISTIE_WKV_SCAN(128, 4, 32);
  } else {
    DISTIE_WKV_SCAN(256, 4, 64);
  }
#undef DISTIE_WKV_SCAN
  return launch_status();
}

extern "C" int distie_wkv_chunk_rows() { return WK_ROWS; }
extern "C" int distie_wkv_chunked_max_dim() { return 128; }

// z: float32 [T, H * D]; chunks: int32 [num_chunks][4] = {request, first row, rows (1..64), 0}, the chunks of a request one
// after the other; request_chunks: int32 [B + 1]; scratch: float32 [num_chunks, H, D, D]; totals: float32 [num_chunks, H, D]
extern "C" int distie_wkv_scan_chunked(const void* r, const void* k, const void* v, const void* gates, int dtype, int64_t ld,
                                       const float* z, const float* bonus, float* state, const float* norm_weight, float eps,
                                       void* out, int out_dtype, float* scratch, float* totals, const int32_t* chunks,
                                       const int32_t* request_chunks, const int32_t* state_slots, int num_chunks, int B,
                                       int H, int D, hipStream_t stream) {
  if (B <= 0 || num_chunks <= 0) return 0;
  if (H < 1 || D < 1 || D > 128 || ld < static_cast<int64_t>(H) * D || !(eps >= 0.f)) return DISTIE_BAD_ARGUMENT;
  const int4* table = reinterpret_cast<const int4*>(chunks);
  const dim3 grid(num_chunks, H);
  const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const int vectors = ld % 4 == 0 && aligned(r) && aligned(k) && aligned(v) && aligned(z) && aligned(scratch) && aligned(bonus) ? 1 : 0;
  int status = 0;
#define DISTIE_WKV_CHUNKS(DP, WHOLE)                                                                                     \
  DISTIE_DISPATCH(dtype, X, DISTIE_DISPATCH(out_dtype, O, {                                                              \
    const bool late = DP <= 64 && static_cast<int64_t>(num_chunks) * H > WK_EARLY_WORKGROUPS;                            \
    const auto outputs = late ? wkv_chunk_outputs_kernel<DP, DP <= 64, WHOLE, X, O>                                      \
                              : wkv_chunk_outputs_kernel<DP, false, WHOLE, X, O>;                                        \
    const int shared = late ? wk_shared<DP, true>() : wk_shared<DP, false>();                                            \
    const int bytes = (WK_ROWS * (DP + 4) + shared + 4 * DP) * static_cast<int>(sizeof(float));                          \
    if (bytes > 48 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(outputs),                                 \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)       \
      return DISTIE_BAD_ARGUMENT;                                                                                        \
    wkv_chunk_sums_kernel<DP, WHOLE, X><<<grid, 256, 0, stream>>>(static_cast<const X*>(k), static_cast<const X*>(v), ld, z,   \
                                                                  scratch, totals, table, H, D);                         \
    if ((status = launch_status()) != 0) return status;                                                                  \
    wkv_chunk_states_kernel<<<dim3(B, H, (D * D + 255) / 256), 256, 0, stream>>>(scratch, totals, state, request_chunks, \
                                                                                state_slots, H, D);                      \
    if ((status = launch_status()) != 0) return status;                                                                  \
    outputs<<<grid, 256, bytes, stream>>>(                                                                               \
        static_cast<const X*>(r), static_cast<const X*>(k), static_cast<const X*>(v), static_cast<const X*>(gates), ld,  \
        z, bonus, scratch, norm_weight, eps, static_cast<O*>(out), table, H, D);                                         \
  }))
#define DISTIE_WKV_WHOLE(DP)             \
  if (vectors && D == DP) {              \
    DISTIE_WKV_CHUNKS(DP, true);         \
  } else {                               \
    DISTIE_WKV_CHUNKS(DP, false);        \
  }
  if (D <= 16) {
    DISTIE_WKV_WHOLE(16);
  } else if (D <= 32) {
    DISTIE_WKV_WHOLE(32);
  } else if (D <= 48) {
    DISTIE_WKV_WHOLE(48);
  } else if (D <= 64) {
    DISTIE_WKV_WHOLE(64);
  } else if (D <= 96) {
    DISTIE_WKV_WHOLE(96);
  } else {
    DISTIE_WKV_WHOLE(128);
  }
#undef DISTIE_WKV_WHOLE
#undef DISTIE_WKV_CHUNKS
  return launch_status();
}

// tanh of a [T, N] float32 view (rows `ld` apart) into a dense tensor
extern "C" int distie_tanh_f32(const float* in, int64_t ld, float* out, int T, int N, hipStream_t stream) {
  if (T <= 0) return 0;
  if (N < 1 || ld < N) return DISTIE_BAD_ARGUMENT;
  const int64_t blocks = (static_cast<int64_t>(T) * N + 255) / 256;
  if (blocks > 0x7fffffff) return DISTIE_BAD_ARGUMENT;
  tanh_f32_kernel<<<static_cast<unsigned>(blocks), 256, 0, stream>>>(in, ld, out, N, T);
  return launch_status();
}
