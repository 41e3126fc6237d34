// Mixture-of-experts feed-forwards: ungated W_down gelu(W_up h) or W_down relu(W_up h)^2, or gated
// W_down (act(W_gate h) * (W_up h)) with [gate rows | up rows] stacked in one weight per expert.
//
// moe_route_scores : softmax over all router outputs, the k largest of score + correction chosen,
//               weights = chosen scores / (their sum + 1e-20) * scale. With groups the outputs form equal groups of
//               neighbours and only those of the best ``keep`` groups (by their largest score + correction) count.
// epilogues of moe_gemm (ACT): 0 none, 1 erf-GELU, 2 tanh-GELU(gate) * up, 3 SiLU(gate) * up, 4 squared ReLU,
//               5 clamped units of gate and up (seqmix_common.h). In the
//               gated forms a workgroup's B tile holds matching gate and up columns, so the product is
//               formed in registers and only F columns are written.
// ids >= E (identity experts) get no tile: moe_group marks their pairs -1 and moe_combine adds
//               w * h for them.
//
// moe_route   : top-k of fp32 router logits (ties to the lower index), softmax over the chosen.
// moe_group   : one workgroup, or two launches of many above 4096 pairs (moe_sort.h), sort the (token, choice)
//               pairs by expert into tiles of 64, 120 or 128 rows (counts and ranks through LDS atomics; a tile holds
//               rows of one expert only).
// moe_tile    : tile GEMM on the matrix cores, bf16 and fp32 (rows of 16-byte pieces); moe_ring: bf16, more than a few rows.
// moe_gemm    : the form for every other size, 64 rows x 64 columns per workgroup, K stepped by 16 through
//               LDS, 4 x 4 outputs per thread. Both: fp32 accumulation in a fixed K order (a row's sums do
//               not depend on its tile or on the rest of the step).
// moe_combine : out[t] = sum_j w[t, j] * y[slot(t, j)] (+ extra[t], a shared expert's row, times sigmoid(g[t]) when it
//               has a gate) in fp32.
#include <algorithm>

#include "moe_ring.h"
#include "moe_tile.h"
#include "seqmix_common.h"
#include "wave_top.h"

using namespace sm;
using namespace moe_tile;

namespace {

constexpr int TM = 64, TN = 64, TK = 16;

__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ logits, int64_t stride, int E, int k,
                                                        int* __restrict__ ids, float* __restrict__ w, int T,
                                                        int sigmoid) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const float* z = logits + t * stride;
  int* oi = ids + (int64_t)t * k;
  float* ow = w + (int64_t)t * k;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY;
    int bi = -1;
    for (int e = 0; e < E; ++e) {
      bool taken = false;
      for (int i = 0; i < j; ++i) taken |= oi[i] == e;
      const float v = z[e];
      if (!taken && (bi < 0 || v > best)) {
        best = v;
        bi = e;
      }
    }
    oi[j] = bi;
    ow[j] = best;
  }
  if (sigmoid) {  // every chosen logit's own sigmoid
    for (int j = 0; j < k; ++j) ow[j] = 1.f / (1.f + expf(-ow[j]));
    return;
  }
  const float m = ow[0];  // the first chosen is the largest
  float s = 0.f;
  for (int j = 0; j < k; ++j) {
    const float p = expf(ow[j] - m);
    ow[j] = p;
    s += p;
  }
  for (int j = 0; j < k; ++j) ow[j] /= s;
}

// One wave per token, lanes over experts (up to NV logits per lane in registers, E <= 512): k rounds
// of a wave-wide arg-max over the logits not yet chosen, ties to the lower index. 64 tokens, 128 experts, 8 chosen: the
// rounds through LDS shuffles took 14 us, now 5 (with scores and groups 6).
template <int NV>
__global__ __launch_bounds__(256) void moe_route_wave_kernel(const float* __restrict__ logits, int64_t stride, int E,
                                                             int k, int* __restrict__ ids, float* __restrict__ w, int T,
                                                             int sigmoid) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= T) return;
  const float* z = logits + t * stride;
  float v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < E ? z[e] : -INFINITY;
  }
  float m0 = 0.f, sum = 0.f, mine = 0.f;  // lane j keeps the j-th chosen weight
  int mine_id = 0;
  unsigned out = wave_top::past_end<NV>(lane, E);
  for (int j = 0; j < k; ++j) {
    const int bi = wave_top::take<NV>(v, out, lane);
    const float best = wave_top::value<NV>(v, bi);
    if (j == 0) m0 = best;
    const float p = sigmoid ? 1.f / (1.f + expf(-best)) : expf(best - m0);
    sum += p;
    if (lane == j) {
      mine = p;
      mine_id = bi;
    }
  }
  if (lane < k) {
    ids[(int64_t)t * k + lane] = mine_id;
    w[(int64_t)t * k + lane] = sigmoid ? mine : mine / sum;
  }
}

// One wave per token, lanes over the router's outputs (E <= 512).
template <int NV>
__global__ __launch_bounds__(256) void moe_route_scores_wave_kernel(const float* __restrict__ logits,
                                                                    const float* __restrict__ corr, int E, int k,
                                                                    int* __restrict__ ids, float* __restrict__ w,
                                                                    int T, int groups, int keep, float scale) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= T) return;
  const float* z = logits + (int64_t)t * E;
  float v[NV], sc[NV], co[NV];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < E ? z[e] : -INFINITY;
    co[i] = e < E ? corr[e] : 0.f;
    mx = fmaxf(mx, v[i]);
  }
  mx = wave_top::largest(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    sc[i] = lane + 64 * i < E ? expf(v[i] - mx) : 0.f;
    sum += sc[i];
  }
  sum = wave_sum(sum);
  unsigned out = wave_top::past_end<NV>(lane, E);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    sc[i] = sc[i] / sum;    // the score
    v[i] = sc[i] + co[i];   // what the choice looks at
  }
  if (groups > 1) {  // groups <= 64: lane g keeps the largest choice score of group g
    const int per = E / groups;
    float gbest = -INFINITY;
    for (int g = 0; g < groups; ++g) {
      float m = -INFINITY;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = lane + 64 * i;
        if (e >= g * per && e < (g + 1) * per) m = fmaxf(m, v[i]);
      }
      m = wave_top::largest(m);
      if (lane == g) gbest = m;
    }
    // a group's rank: how many are larger, or equal with a lower index
    int rank = 0;
    for (int g = 0; g < groups; ++g) {
      const float o = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gbest), g));
      rank += (o > gbest || (o == gbest && g < lane)) ? 1 : 0;
    }
    const uint64_t kept = __ballot(lane < groups && rank < keep);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = lane + 64 * i;
      if (e < E && !(kept >> (e / per) & 1ull)) out |= 1u << i;
    }
  }
  float wsum = 0.f, mine = 0.f;
  int mine_id = 0;
  for (int j = 0; j < k; ++j) {
    const int bi = wave_top::take<NV>(v, out, lane);
    const float best = wave_top::value<NV>(sc, bi);
    wsum += best;
    if (lane == j) {
      mine = best;
      mine_id = bi;
    }
  }
  if (lane < k) {
    ids[(int64_t)t * k + lane] = mine_id;
    w[(int64_t)t * k + lane] = mine / (wsum + 1e-20f) * scale;
  }
}

// Any E: one thread per token.
__global__ __launch_bounds__(256) void moe_route_scores_kernel(const float* __restrict__ logits,
                                                               const float* __restrict__ corr, int E, int k,
                                                               int* __restrict__ ids, float* __restrict__ w, int T,
                                                               int groups, int keep, float scale) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const float* z = logits + (int64_t)t * E;
  int* oi = ids + (int64_t)t * k;
  float* ow = w + (int64_t)t * k;
  float mx = -INFINITY, sum = 0.f;
  for (int e = 0; e < E; ++e) mx = fmaxf(mx, z[e]);
  for (int e = 0; e < E; ++e) sum += expf(z[e] - mx);
  const int per = E / groups;
  auto group_best = [&](int g) {
    float m = -INFINITY;
    for (int e = g * per; e < (g + 1) * per; ++e) m = fmaxf(m, expf(z[e] - mx) / sum + corr[e]);
    return m;
  };
  // the last group kept: one after the other in falling order, ties to the lower index
  float last = INFINITY;
  int last_g = -1;
  if (groups > 1) {
    for (int n = 0; n < keep; ++n) {
      float best = -INFINITY;
      int bg = -1;
      for (int g = 0; g < groups; ++g) {
        const float m = group_best(g);
        const bool after = m < last || (m == last && g > last_g);
        if (after && (bg < 0 || m > best)) {
          best = m;
          bg = g;
        }
      }
      last = best;
      last_g = bg;
    }
  }
  float wsum = 0.f;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY, bsc = 0.f;
    int bi = -1;
    for (int e = 0; e < E; ++e) {
      if (groups > 1 && e % per == 0) {
        const float m = group_best(e / per);
        if (m < last || (m == last && e / per > last_g)) {  // not kept
          e += per - 1;
          continue;
        }
      }
      bool taken = false;
      for (int i = 0; i < j; ++i) taken |= oi[i] == e;
      const float sc = expf(z[e] - mx) / sum;
      const float c = sc + corr[e];
      if (!taken && (bi < 0 || c > best)) {
        best = c;
        bsc = sc;
        bi = e;
      }
    }
    oi[j] = bi;
    ow[j] = bsc;
    wsum += bsc;
  }
  for (int j = 0; j < k; ++j) ow[j] = ow[j] / (wsum + 1e-20f) * scale;
}

// C[slot, n] = act(sum_k A[row(slot), k] * W[e, n, k]);  row(slot) = pair / kdiv (gathered
// tokens) when kdiv > 0, the slot itself otherwise.
__device__ __forceinline__ float gelu_erf_(float v) { return 0.5f * v * (1.f + erff(v * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_tanh_(float v) {
  return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
}
constexpr bool gated_act_code(int act) { return act == 2 || act == 3 || act == 5; }
template <typename T, int ACT>
__device__ __forceinline__ float gated_(float g, float u, float limit) {
  if (ACT == 5) return clamped_unit<T>(g, u, limit);
  return (ACT == 2 ? gelu_tanh_(g) : g / (1.f + expf(-g))) * u;
}

// Gated forms (ACT 2, 3 and 5): N is the number of OUTPUT columns F; the weight has 2 N rows [gate | up].
// The workgroup's 64 B rows are 32 gate rows n0.. and the 32 matching up rows; a thread's four
// columns are two gate columns and their two up columns.
template <typename T, int ACT>
__global__ __launch_bounds__(256) void moe_gemm_kernel(const T* __restrict__ A, int64_t a_stride, int kdiv,
                                                       const int* __restrict__ slot_row,
                                                       const int* __restrict__ tiles, const T* __restrict__ Wt,
                                                       int N, int K, T* __restrict__ Cout,
                                                       const float* __restrict__ row_w, float limit) {
  if ((int)blockIdx.x >= tiles[0]) return;
  const int e = tiles[1 + 3 * blockIdx.x] & 0xffff, rows = tiles[1 + 3 * blockIdx.x] >> 16;
  __shared__ float sA[TK][TM + 4], sB[TK][TN + 4];
  __shared__ int srow[TM];
  __shared__ float sw[TM];  // the row's input weight (gated forms with row_w): scales both sums
  const int tid = threadIdx.x;
  constexpr bool GATED = gated_act_code(ACT);
  const int slot0 = blockIdx.x * TM, n0 = blockIdx.y * (GATED ? TN / 2 : TN);
  if (tid < TM) {
    const int p = tid < rows ? slot_row[slot0 + tid] : -1;
    srow[tid] = p < 0 ? -1 : (kdiv > 0 ? p / kdiv : slot0 + tid);
    sw[tid] = (row_w != nullptr && p >= 0) ? row_w[p] : 1.f;
  }
  __syncthreads();
  const T* We = Wt + (int64_t)e * (GATED ? 2 * N : N) * K;
  const int lr = tid >> 2, lk = (tid & 3) * 4;  // loader: row / column lr, 4 consecutive k
  const int ty = tid >> 4, tx = tid & 15;       // compute: rows ty*4.., columns tx*4.. (gated: see above)
  float acc[4][4] = {};
  const int arow = srow[lr];
  const int bcol = GATED ? n0 + (lr & 31) : n0 + lr;          // output column this B row belongs to
  const int brow = GATED && lr >= 32 ? N + bcol : bcol;         // its row in the expert's weight
  for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = k0 + lk + i;
      sA[lk + i][lr] = (arow >= 0 && kk < K) ? ld(A + (int64_t)arow * a_stride + kk) : 0.f;
      sB[lk + i][lr] = (bcol < N && kk < K) ? ld(We + (int64_t)brow * K + kk) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = sA[kk][ty * 4 + i];
        b[i] = GATED ? sB[kk][(i >> 1) * 32 + tx * 2 + (i & 1)] : sB[kk][tx * 4 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (srow[r] < 0) continue;
    if (GATED) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + tx * 2 + j;
        if (n < N) st(Cout + (int64_t)(slot0 + r) * N + n, gated_<T, ACT>(sw[r] * acc[i][j], sw[r] * acc[i][j + 2], limit));
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (ACT == 1) v = gelu_erf_(v);
      if (ACT == 4) {
        v = fmaxf(v, 0.f);
        v *= v;
      }
      st(Cout + (int64_t)(slot0 + r) * N + n, v);
    }
  }
}


template <typename T> __device__ __forceinline__ void put4(void* o, const float (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x4_t*>(o) = f32x4_t{v[0], v[1], v[2], v[3]};
  } else {
    ushort4 b;
    st(&b.x, v[0]); st(&b.y, v[1]); st(&b.z, v[2]); st(&b.w, v[3]);
    *reinterpret_cast<ushort4*>(o) = b;
  }
}

template <typename T, int ACT>
__device__ __forceinline__ void finish4(float (&v)[4], const f32x4_t& g, const f32x4_t& u, float sw, float limit) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v[q] = g[q];
    if (gated_act_code(ACT)) v[q] = gated_<T, ACT>(sw * g[q], sw * u[q], limit);
    if (ACT == 1) v[q] = gelu_erf_(v[q]);
    if (ACT == 4) {
      v[q] = fmaxf(v[q], 0.f);
      v[q] *= v[q];
    }
  }
}

template <typename T, int ACT>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(const T* __restrict__ A, int64_t a_stride, int kdiv,
                                                          const int* __restrict__ slot_row, const int* __restrict__ tiles,
                                                          const T* __restrict__ Wt, int N, int K, T* __restrict__ Cout,
                                                          const float* __restrict__ row_w, float limit, int NB, int tm, const int* __restrict__ order) {
  constexpr bool GATED = gated_act_code(ACT);
  Work wk;
  if (order != nullptr ? !find_work_by_size(tiles, order, NB, wk) : !find_work(tiles, NB, wk)) return;
  const int nb = wk.nb, tile = wk.tile, e = wk.e, rows = wk.rows;
  __shared__ __attribute__((aligned(128))) char lds[sizeof(T) == 4 ? SLDS : 4 * TBUF];
  const int tid = threadIdx.x;
  const int64_t slot0 = (int64_t)tile * tm;
  const int col0 = nb * (GATED ? TBW / 2 : TBW);  // the workgroup's first output column
  MoeTile t;
  t.K = K, t.lds = lds, t.w = reinterpret_cast<const char*>(Wt + (int64_t)e * (GATED ? 2 * N : N) * K);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // slots past the tile's rows read its last row: their sums are not stored
    const int r = min((tid >> 3) + i * 32, rows - 1);
    const int64_t src = kdiv > 0 ? slot_row[slot0 + r] / kdiv : slot0 + r;
    t.ap[i] = reinterpret_cast<const char*>(A + src * a_stride) + (tid & 7) * 16;
  }
  // columns past N read the last one and are not stored either
  auto wrow = [&](int j) {
    const int col = min(col0 + (GATED ? j & 63 : j), N - 1);
    return (uint32_t)(col + (GATED && j >= 64 ? N : 0)) * (uint32_t)(K * (int)sizeof(T));
  };
  auto out = [&](int r, int c, const f32x4_t& g, const f32x4_t& u) {
    if (r >= rows) return;
    float sw = 1.f;  // the row's input weight (gated forms with row_w): scales both sums
    if (GATED && row_w != nullptr) sw = row_w[slot_row[slot0 + r]];
    float v[4];
    finish4<T, ACT>(v, g, u, sw, limit);
    T* o = Cout + (slot0 + r) * N;
    const int n = col0 + c;
    if (n + 4 <= N && (N & 3) == 0) {
      put4<T>(o + n, v);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < N) st(o + n + q, v[q]);
    }
  };
  run_tile<T, GATED>(t, rows, wrow, out);
}

// bf16 steps that bring an expert more than a few rows (moe_ring.h).
template <int ACT>
__global__ __launch_bounds__(moe_ring::NT, 2) void moe_ring_kernel(const bf16_t* __restrict__ A, int64_t a_stride, int kdiv,
                                                                     const int* __restrict__ slot_row,
                                                                     const int* __restrict__ tiles, const bf16_t* __restrict__ Wt,
                                                                     int N, int K, bf16_t* __restrict__ Cout,
                                                                     const float* __restrict__ row_w, float limit) {
  __shared__ __attribute__((aligned(1024))) char lds[moe_ring::LDS];
  constexpr bool GATED = gated_act_code(ACT);
  // the row's input weight scales both sums
  auto scale = [&](int64_t slot) { return GATED && row_w != nullptr ? row_w[slot_row[slot]] : 1.f; };
  auto act = [&](float g, float u, float sw) {
    if constexpr (GATED) return gated_<bf16_t, ACT>(sw * g, sw * u, limit);
    if (ACT == 1) return gelu_erf_(g);
    if (ACT == 4) {
      g = fmaxf(g, 0.f);
      return g * g;
    }
    return g;
  };
  moe_ring::run<GATED ? moe_ring::HALVES : moe_ring::PLAIN>(A, a_stride, kdiv, slot_row, tiles, Wt, N, K, Cout, scale, act, lds);
}

template <typename T>
__global__ __launch_bounds__(256) void moe_combine_kernel(const T* __restrict__ y, const int* __restrict__ pair_slot,
                                                          const float* __restrict__ w, int k, int d,
                                                          T* __restrict__ out, const T* __restrict__ h,
                                                          const T* __restrict__ extra,
                                                          const float* __restrict__ eg, int64_t eg_stride) {
  const int64_t t = blockIdx.x;
  const float ge = eg ? 1.f / (1.f + expf(-eg[t * eg_stride])) : 1.f;
  for (int c = threadIdx.x; c < d; c += 256) {
    float s = 0.f;
    for (int j = 0; j < k; ++j) {
      const int slot = pair_slot[t * k + j];
      // slot < 0: an identity expert returns the token's own input
      s += (w ? w[t * k + j] : 1.f) * (slot >= 0 ? ld(y + (int64_t)slot * d + c) : ld(h + t * d + c));
    }
    if (extra) s += ge * ld(extra + t * d + c);
    st(out + t * d + c, s);
  }
}

// Rows of whole groups of eight: a thread sums eight columns from 16-byte loads. Bound by the rows' way from memory:
// 700 tokens of 8 fp32 rows of 2048 (46 MB) 38 us by elements, here 13; 2048 tokens in bf16 15.7.
__device__ __forceinline__ void fma8(float (&s)[8], float w, const bf16_t* p) {
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] += w * __uint_as_float((v[q >> 1] >> (16 * (q & 1))) << 16);
}
__device__ __forceinline__ void fma8(float (&s)[8], float w, const float* p) {
  const f32x4_t v[2] = {*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 4)};
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] += w * v[q >> 2][q & 3];
}
__device__ __forceinline__ void put8(bf16_t* p, const float (&s)[8]) {
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const __bf16 a = (__bf16)s[2 * q], b = (__bf16)s[2 * q + 1];
    o[q] = (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
  }
  *reinterpret_cast<u32x4_t*>(p) = o;
}
__device__ __forceinline__ void put8(float* p, const float (&s)[8]) {
  *reinterpret_cast<f32x4_t*>(p) = f32x4_t{s[0], s[1], s[2], s[3]};
  *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{s[4], s[5], s[6], s[7]};
}
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(const T* __restrict__ y, const int* __restrict__ pair_slot,
                                                              const float* __restrict__ w, int k, int d, T* __restrict__ out,
                                                              const T* __restrict__ h, const T* __restrict__ extra,
                                                              const float* __restrict__ eg, int64_t eg_stride) {
  const int64_t t = blockIdx.x;
  const float ge = eg ? 1.f / (1.f + expf(-eg[t * eg_stride])) : 1.f;
  for (int c = threadIdx.x * 8; c < d; c += 256 * 8) {
    float s[8] = {};
    for (int j = 0; j < k; ++j) {
      const int slot = pair_slot[t * k + j];
      fma8(s, w ? w[t * k + j] : 1.f, slot >= 0 ? y + (int64_t)slot * d + c : h + t * d + c);
    }
    if (extra) fma8(s, ge, extra + t * d + c);
    put8(out + t * d + c, s);
  }
}

// Router logits: y = x W^T in fp32 from bf16 rows and weights. Their products are exact in fp32, so the fp32 matrix instructions on
// widened operands give what a product of float copies gave, without the copies: a lane's four neighbouring k of a step of 16 are
// the operands of four instructions, which is also the order in which the float product that stood here added (the same bits
// at 1 .. 800 x (132, 2048)).
// Bound by the instructions' chain (one waits 75 cycles for the one before): four waves per 16 x 16 numbers, which take 32 k of every 128
// each and are added up in order. Chunks of 128 k come to LDS two ahead, in 16-byte pieces whose place in a row is turned by the row's
// number: the eight bytes that a lane takes then lie in banks of their own.
// us, copy and float product / here: 1 x (132, 2048) 11.2 / 9.2, 64 12.3 / 9.2, 700 16.1 / 11.3, 800 x (64, 1024) 13.1 / 6.3; up to 511 such blocks
// and K 2048: 64 x (128, 4096) 14.3 / 15.0; 2048 x (132, 2048) in the order of its float product, one chain of all k, 34.1 / 28.9,
// but 1500 24.1 / 28.2 and 2722 33.7 / 37.3.
constexpr int RCH = 128, RROW = RCH * 2, RBLK = 16 * RROW, RSTAGE = 2 * RBLK;  // k of a chunk, bytes of a row, of 16 rows, of both operands
template <int N>
__device__ __forceinline__ void router_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

__global__ __launch_bounds__(256) void router_kernel(const bf16_t* __restrict__ x, int64_t xs, const bf16_t* __restrict__ w, int M,
                                                     int N, int K, int nb, float* __restrict__ y) {
  __shared__ __attribute__((aligned(16))) char ring[3 * RSTAGE];  // 16 rows of x, then 16 of w
  __shared__ __attribute__((aligned(16))) f32x4_t red[3][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  const int m0 = blockIdx.x / nb * 16, n0 = blockIdx.x % nb * 16;
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring + wave * 1024;
  // a wave's copy of 1 KB is four rows: lane l's 16 bytes are piece (l % 16) ^ row of row 4 wave + l / 16
  const int row = 4 * wave + (lane >> 4), piece = ((lane & 15) ^ row) * 16;
  const uint32_t xo = (uint32_t)((min(m0 + row, M - 1) - m0) * xs * 2) + piece;
  const uint32_t wo = (uint32_t)((min(n0 + row, N - 1) - n0) * (int64_t)K * 2) + piece;
  const char* xb = (const char*)(x + m0 * xs);
  const char* wb = (const char*)(w + (int64_t)n0 * K);
  const auto fetch = [&](int c) {
    const uint32_t at = lds + c % 3 * RSTAGE;
    copy_1k(xb + (int64_t)c * RROW, xo, at);
    copy_1k(wb + (int64_t)c * RROW, wo, at + RBLK);
  };
  int at[2];  // of the wave's two steps of 16 k in a chunk
#pragma unroll
  for (int b = 0; b < 2; ++b) at[b] = r16 * RROW + ((4 * wave + 2 * b + (g >> 1)) ^ r16) * 16 + 8 * (g & 1);
  const int chunks = K / RCH;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  fetch(0);
  if (chunks > 1) fetch(1);
  for (int c = 0; c < chunks; ++c) {
    if (c + 1 == chunks) router_wait<0>();
    else router_wait<2>();
    __builtin_amdgcn_s_barrier();  // chunk c is there, chunk c - 1 no longer read
    asm volatile("" ::: "memory");
    if (c + 2 < chunks) fetch(c + 2);
    const char* t = ring + c % 3 * RSTAGE;
    uint2 a[2], q[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      a[b] = *reinterpret_cast<const uint2*>(t + at[b]);
      q[b] = *reinterpret_cast<const uint2*>(t + RBLK + at[b]);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t av[4] = {a[b].x << 16, a[b].x & 0xffff0000u, a[b].y << 16, a[b].y & 0xffff0000u};
      const uint32_t qv[4] = {q[b].x << 16, q[b].x & 0xffff0000u, q[b].y << 16, q[b].y & 0xffff0000u};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(qv[j]), __uint_as_float(av[j]), acc, 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads of the chunk are done
  }
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < 3; ++i) acc += red[i][lane];
  // acc[r] = y[m0 + r16][n0 + 4 g + r]
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (m0 + r16 < M && n0 + 4 * g + r < N) y[(int64_t)(m0 + r16) * N + n0 + 4 * g + r] = acc[r];
}

}  // namespace

extern "C" {

// sigmoid: the weights are the chosen logits' sigmoids instead of the softmax over the chosen logits.
// stride: between the rows of the logits (they may be the first E columns of a wider product).
void sm_moe_route(const float* logits, int64_t stride, int E, int k, int* ids, float* w, int T, int sigmoid,
                  hipStream_t stream) {
  if (T == 0) return;
  if (E <= 512 && k <= 64) {
#define SM_GO(NV) \
  hipLaunchKernelGGL(moe_route_wave_kernel<NV>, dim3((T + 3) / 4), dim3(256), 0, stream, logits, stride, E, k, ids, w, T, sigmoid)
    if (E <= 64) SM_GO(1);
    else if (E <= 128) SM_GO(2);
    else if (E <= 256) SM_GO(4);
    else SM_GO(8);
#undef SM_GO
    return;
  }
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 255) / 256), dim3(256), 0, stream, logits, stride, E, k, ids, w, T,
                     sigmoid);
}

// x [M, K] bf16 rows xs apart, w [N, K], y [M, N] fp32. -1: not these operands
int sm_router(const void* x, int64_t xs, const void* w, int M, int N, int K, float* y, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  if (K < RCH || K % RCH || K > 2048 || xs % 8 || xs < 0 || xs > (1 << 24) || (((uintptr_t)x | (uintptr_t)w) & 15) || M > 8192 || N > 8192)
    return -1;
  const int nb = (N + 15) / 16, blocks = (M + 15) / 16 * nb;
  if (blocks >= 512) return -1;
  hipLaunchKernelGGL(router_kernel, dim3(blocks), dim3(256), 0, stream, (const bf16_t*)x, xs, (const bf16_t*)w, M, N, K, nb, y);
  return 0;
}

void sm_moe_route_scores(const float* logits, const float* corr, int E, int k, int* ids, float* w, int T, int groups,
                         int keep, float scale, hipStream_t stream) {
  if (T == 0) return;
  if (E <= 512 && k <= 64 && groups <= 64) {
#define SM_GO(NV)                                                                                                          \
  hipLaunchKernelGGL(moe_route_scores_wave_kernel<NV>, dim3((T + 3) / 4), dim3(256), 0, stream, logits, corr, E, k, ids, w, T, \
                     groups, keep, scale)
    if (E <= 64) SM_GO(1);
    else if (E <= 128) SM_GO(2);
    else if (E <= 256) SM_GO(4);
    else SM_GO(8);
#undef SM_GO
    return;
  }
  hipLaunchKernelGGL(moe_route_scores_kernel, dim3((T + 255) / 256), dim3(256), 0, stream, logits, corr, E, k, ids, w,
                     T, groups, keep, scale);
}

// Counters that a sort of n pairs over E experts needs as scratch.
int64_t sm_moe_sort_scratch(int n, int E) { return moe_sort::many(n, E) ? (int64_t)moe_sort::blocks(n) * E : 0; }

// order: null, or where the tiles are listed by size.
void sm_moe_group(const int* ids, int n, int E, int tm, int* hist, int* slot_row, int* tiles, int* pair_slot,
                  int* order, hipStream_t stream) {
  launch_group(ids, n, E, tm, hist, slot_row, tiles, pair_slot, order, stream);
}

// Which tile (its place by size) and block of weight rows a workgroup of the form by size takes.
void sm_moe_deal(int total, int NB, int block, int* rank, int* nb) {
  const Dealt d = deal(total, NB, block);
  *rank = d.rank, *nb = d.nb;
}

// Whether the matrix-core form takes these operands: 16-byte pieces of every row, an expert (``rows`` weight rows) within
// 32-bit offsets. Its tiles have 128 slots, the other form's 64.
int sm_moe_tiled(const void* A, int64_t a_stride, const void* W, int64_t rows, int64_t K, int f32) {
  const int per = f32 ? 4 : 8;
  return K % per == 0 && rows * K * (f32 ? 4 : 2) < (int64_t)1 << 32 && a_stride % per == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0;
}

// Whether the form of many rows takes them: bf16, whole steps of K, whole 16-byte pieces of the output rows (``rows`` weight
// rows, half of them columns in the gated forms), byte offsets below 2^31.
int sm_moe_ring(const void* A, int64_t a_rows, int64_t a_stride, const void* W, int64_t rows, int64_t K, int gated, int f32) {
  return !f32 && sm_moe_tiled(A, a_stride, W, rows, K, 0) && K % 64 == 0 && K >= 256 && rows % (gated ? 16 : 8) == 0 &&
         rows * K * 2 < (int64_t)1 << 31 && a_stride >= 0 && a_rows * a_stride * 2 < (int64_t)1 << 31;
}

// act: 0 none, 1 erf-GELU, 2 tanh-GELU(gate) * up, 3 SiLU(gate) * up, 4 squared ReLU, 5 clamped units. N = output
// columns (the gated forms read a weight of 2 N rows per expert). tm: slots per tile, 120 or 128 for the matrix-core form (operands
// that sm_moe_tiled takes), 64 for the other. ring: the form of many rows (sm_moe_ring), tiles of 120. Where only one of a step's
// two products has the sizes for it, the other takes the tiles of 120 in moe_tile_kernel: 128 experts of 2048 x 720, 8 chosen,
// both products with sorting and sum, us, neither in it / one: 24 rows 272 / 255, 62 rows 334 / 315, 256 rows 644 / 601; of 2056 x 768,
// 24 rows 299 / 287, 256 rows 832 / 676.
// by_size (tiles of 128 rows): behind the tables the tiles' order (sm_moe_group), in which they are taken.
// row_w (gated forms): fp32 weight per (token, choice) pair that scales the row's INPUT, applied to
// both fp32 sums before the activation; nullptr = 1.
void sm_moe_gemm(const void* A, int64_t a_stride, int kdiv, const int* slot_row, const int* tiles, const void* W,
                 int N, int K, void* C, int max_tiles, int tm, int ring, int by_size, int act, int f32, const float* row_w,
                 float limit, hipStream_t stream) {
  const bool gated = gated_act_code(act);
  if (ring) {
    const int cols = gated ? moe_ring::WROWS / 2 : moe_ring::WROWS;
    const int64_t items = (int64_t)max_tiles * ((N + cols - 1) / cols);
    const dim3 grid((unsigned)std::min<int64_t>((items + 7) / 8 * 8, 512));  // two workgroups per CU
#define SM_RING(A_)                                                                                                        \
  hipLaunchKernelGGL(moe_ring_kernel<A_>, grid, dim3(moe_ring::NT), 0, stream, (const bf16_t*)A, a_stride, kdiv, slot_row, \
                     tiles, (const bf16_t*)W, N, K, (bf16_t*)C, row_w, limit)
    if (act == 0) SM_RING(0);
    else if (act == 1) SM_RING(1);
    else if (act == 2) SM_RING(2);
    else if (act == 3) SM_RING(3);
    else if (act == 4) SM_RING(4);
    else SM_RING(5);
#undef SM_RING
    return;
  }
  if (tm != TM) {
    const int NB = (N + (gated ? 63 : 127)) / (gated ? 64 : 128);
    const int64_t items = (int64_t)max_tiles * NB;
    const int* order = by_size ? tiles + 1 + 3 * (int64_t)max_tiles : nullptr;
    const dim3 grid((unsigned)(by_size ? (int64_t)((max_tiles + 7) / 8 * 8) * NB : (items + 7) / 8 * 8));
#define SM_MT(KERN, TYPE, GRID)                                                                                       \
  hipLaunchKernelGGL(KERN, GRID, dim3(256), 0, stream, (const TYPE*)A, a_stride, kdiv, slot_row, tiles, (const TYPE*)W, \
                     N, K, (TYPE*)C, row_w, limit, NB, tm, order)
#define SM_MT2(A_)                                                                  \
  if (f32) SM_MT((moe_tile_kernel<float, A_>), float, grid);                        \
  else SM_MT((moe_tile_kernel<bf16_t, A_>), bf16_t, grid)
    if (act == 0) { SM_MT2(0); }
    else if (act == 1) { SM_MT2(1); }
    else if (act == 2) { SM_MT2(2); }
    else if (act == 3) { SM_MT2(3); }
    else if (act == 4) { SM_MT2(4); }
    else { SM_MT2(5); }
#undef SM_MT2
#undef SM_MT
    return;
  }
  const int tn = gated ? TN / 2 : TN;
  const dim3 grid(max_tiles, (N + tn - 1) / tn);
#define SM_GO(TYPE, A_)                                                                                         \
  hipLaunchKernelGGL((moe_gemm_kernel<TYPE, A_>), grid, dim3(256), 0, stream, (const TYPE*)A, a_stride, kdiv,   \
                     slot_row, tiles, (const TYPE*)W, N, K, (TYPE*)C, row_w, limit)
#define SM_GO2(TYPE)                   \
  if (act == 0) SM_GO(TYPE, 0);        \
  else if (act == 1) SM_GO(TYPE, 1);   \
  else if (act == 2) SM_GO(TYPE, 2);   \
  else if (act == 3) SM_GO(TYPE, 3);   \
  else if (act == 4) SM_GO(TYPE, 4);   \
  else SM_GO(TYPE, 5)
  if (f32) { SM_GO2(float); }
  else { SM_GO2(bf16_t); }
#undef SM_GO2
#undef SM_GO
}

// extra [T, d] with its gate logits eg (fp32, row stride eg_stride; null: no gate): a shared expert's rows, or null.
void sm_moe_combine(const void* y, const int* pair_slot, const float* w, int k, int d, void* out, const void* h, int T,
                    int f32, const void* extra, const float* eg, int64_t eg_stride, hipStream_t stream) {
  if (T == 0) return;
#define SM_CO(KERN, TYPE)                                                                                       \
  hipLaunchKernelGGL(KERN, dim3(T), dim3(256), 0, stream, (const TYPE*)y, pair_slot, w, k, d, (TYPE*)out,       \
                     (const TYPE*)h, (const TYPE*)extra, eg, eg_stride)
  const bool vec = d % 8 == 0 && (((uintptr_t)y | (uintptr_t)out | (uintptr_t)h | (uintptr_t)extra) & 15) == 0;
  if (f32 && vec) SM_CO(moe_combine_vec_kernel<float>, float);
  else if (f32) SM_CO(moe_combine_kernel<float>, float);
  else if (vec) SM_CO(moe_combine_vec_kernel<bf16_t>, bf16_t);
  else SM_CO(moe_combine_kernel<bf16_t>, bf16_t);
#undef SM_CO
}

}  // extern "C"
