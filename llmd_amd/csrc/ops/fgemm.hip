// fp32 products y[M, N] = x[M, K] . w[N, K]^T (+ bias) of prompt-sized steps on the bf16 matrix units: every number, times 2^24, is the
// exact sum of three bf16 parts, and the six largest of the nine products of parts are formed in fp32 sums (what is left out is at most
// 2^-24 of a product: moe_tile.h, which has the same for experts), the largest ones in sums of their own, so that a sum is rounded once
// per 32 products.
//
// What bounds it: 96 products of parts (16 cycles each) and some 230 vector instructions to scale and split the next numbers, of which a
// SIMD takes two beside a product without losing time, per 128 x 128 x 32: 1536 cycles at least, 2300 measured without the scaling,
// which costs 2 to 3 % (700 x (3072, 2048) 59.8 / 61.6 us, 2048 x (5120, 2048) 240 / 246). Each number is
// split once per workgroup, on its way from registers to LDS; the splitting, LDS reads and loads lie between the products in
// the order they are written here. Three buffers of LDS: a step's first operands are read beside the step before it.
//
// us, vendor library / here: 700 x (5120, 2048) 152 / 81, (2048, 4096) 98 / 78, (3072, 2048) 103 / 55, (2048, 1536) 56 / 35;
// 2048 x (5120, 2048) 302 / 238. Off 64 bits, relative, any of these sizes: K 512 4.0e-7 / 1.3e-7, 2048 4.1e-7 / 2.7e-7, 4096 5.7e-7 /
// 4.0e-7.
#include <algorithm>
#include <cmath>

#include "llmd_common.h"
#include "moe_tile.h"

using namespace moe_tile;

namespace {

constexpr int BK = 32;
constexpr int MARK = 4 * TBUF;  // rows of the tile that fp32 instructions form: behind what moe_tile_many uses

constexpr int plane(int rows) { return rows * BK * 2; }
constexpr int lds_bytes(int mi, int ni) { return std::max(3 * 3 * plane(32 * (mi + ni)), MARK + TBM * 4); }

// the accumulator tied to AGPRs: hipcc re-homes loop-carried accumulators of the builtin every iteration
__device__ __forceinline__ void acc_mma(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// f(0), f(1), .. f(N - 1), the numbers as types
template <typename F, int... J>
__device__ __forceinline__ void each_(F& f, std::integer_sequence<int, J...>) {
  (f(Set<J>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F f) {
  each_(f, std::make_integer_sequence<int, N>{});
}

// Tile of 32 MI x 32 NI, four waves of 16 MI x 16 NI. Rows past the end read the last one.
template <int MI, int NI>
__global__ __launch_bounds__(256, 1) void fgemm_kernel(const float* __restrict__ x, int64_t ldx,
                                                                         const float* __restrict__ w, int64_t ldw,
                                                                         float* __restrict__ y, int64_t ldy, int M, int N,
                                                                         int K, const float* __restrict__ bias, int ranges) {
  constexpr int BM = 32 * MI, BN = 32 * NI, NP = (MI + NI) / 2;  // passes of 64 rows of the tile's x, then w
  constexpr int PL = plane(BM + BN), BUF = 3 * PL;
  static_assert((MI + NI) % 2 == 0, "passes of 64 rows");
  __shared__ __attribute__((aligned(128))) char lds[lds_bytes(MI, NI)];
  const int tiles = (M + BM - 1) / BM;
  int item = llmd::xcd_remap(blockIdx.x, gridDim.x);
  if (ranges > 1) {  // sums of a range of K: y is [ranges, M, N]
    const int all = tiles * ((N + BN - 1) / BN), range = item / all, chunk = (K / BK + ranges - 1) / ranges * BK;
    item -= range * all;
    x += range * chunk;
    w += range * chunk;
    y += (int64_t)range * M * ldy;
    K = range + 1 < ranges ? chunk : K - range * chunk;
  }
  const int m0 = item % tiles * BM, n0 = item / tiles * BN;
  const int rows = min(M - m0, BM), cols = min(N - n0, BN);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  const int wr = wave >> 1, wc = wave & 1;
  const int nk = K / BK;

  // this thread's 8 of a step's 32 elements of row (tid >> 2) + 64 p; rows past the end read the last one
  const float* src[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int r = 64 * p + (tid >> 2);
    src[p] = (r < BM ? x + (m0 + min(r, rows - 1)) * ldx : w + (n0 + min(r - BM, cols - 1)) * ldw) + (tid & 3) * 8;
  }
  const auto place = [](int row, int q) { return row * 64 + ((q ^ ((0x1E >> (2 * (row >> 2 & 3))) & 3)) * 16); };
  const int st = place(tid >> 2, tid & 3);
  const int ra = place(wr * 16 * MI + r16, kq), rw = place(BM + wc * 16 * NI + r16, kq);

  // part o of a pair of elements: their rounding to bf16 (two numbers in v), and what is left of each
  f32x4_t g[2][NP][2];
  uint32_t v[3][4];
  auto load = [&](int s, int p, int h, int kt) { g[s][p][h] = reinterpret_cast<const f32x4_t*>(src[p] + min(kt, nk - 1) * BK)[h]; };
  auto part = [&](int s, int p, int pair, int o) {
    float* x = reinterpret_cast<float*>(&g[s][p][pair >> 1]) + 2 * (pair & 1);
    if (o == 0) x[0] *= SPLIT_UP, x[1] *= SPLIT_UP;
    asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(v[o][pair]) : "v"(x[0]), "v"(x[1]));
  };
  auto rest = [&](int s, int p, int pair, int o, int h) {
    float* x = reinterpret_cast<float*>(&g[s][p][pair >> 1]) + 2 * (pair & 1);
    x[h] -= __uint_as_float(h ? v[o][pair] & 0xffff0000u : v[o][pair] << 16);
  };
  auto put = [&](char* buf, int p, int o) {
    *reinterpret_cast<u32x4_t*>(buf + o * PL + st + p * 4096) = u32x4_t{v[o][0], v[o][1], v[o][2], v[o][3]};
  };
  constexpr int PER = 33, PI = 57, U = PER * NP, S = 6 * MI * NI;  // side works and instructions of a pass; works, products of a step
  // instructions before side work u
  constexpr auto before = [](int u) {
    const int q = u % PER, r = q % 13, first = q < 13 ? 3 : 1;  // (a pair's first part: two products and the rounding)
    return u / PER * PI + (q >= 26 ? 50 + q - 26 : q / 13 * 29 + (r < 4 ? first * r : 4 * first + 2 * (r - 4)));
  };
  constexpr auto first_at = [before](int n) {  // the first side work from product n on
    int u = 0;
    while (u < U && before(u) * S < n * (NP * PI)) ++u;
    return u;
  };
  // side work u: the pass's 4 pairs split part by part, each part's 16 bytes to LDS, the pass's next loads
  auto side = [&](auto u_, int s, char* buf, int kt) {
    constexpr int u = decltype(u_)::value, p = u / PER, q = u % PER;
    if constexpr (q >= 31) load(s, p, q - 31, kt);
    else if constexpr (q == 30) put(buf, p, 2);
    else if constexpr (q >= 26) part(s, p, q - 26, 2);
    else if constexpr (q % 13 < 4) part(s, p, q % 13, q / 13);
    else if constexpr (q % 13 < 12) rest(s, p, (q % 13 - 4) >> 1, q / 13, q & 1 ^ (q / 13 & 1));
    else put(buf, p, q / 13);
  };
  f32x4_t big[MI][NI], small[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) big[i][j] = small[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wf[2][NI][3], af[2][3];  // the step's and the next one's weights, two blocks' rows
  auto read_w = [&](int set, const char* buf, int n) { wf[set][n / 3][n % 3] = *reinterpret_cast<const u32x4_t*>(buf + n % 3 * PL + rw + n / 3 * 1024); };
  auto read_a = [&](int set, const char* buf, int i, int o) { af[set][o] = *reinterpret_cast<const u32x4_t*>(buf + o * PL + ra + i * 1024); };
  auto product = [&](auto set_, auto n_) {
    constexpr int PW[6] = {0, 0, 1, 1, 0, 2}, PA[6] = {0, 1, 0, 1, 2, 0}, set = decltype(set_)::value, n = decltype(n_)::value;
    constexpr int i = n / (6 * NI), k = 5 - n / NI % 6, j = n % NI;  // the smallest products first
    acc_mma(k == 0 ? big[i][j] : small[i][j], wf[set][j][PW[k]], af[(set * MI + i) & 1][PA[k]]);
  };

  char* cur = lds;
  // step kt, its first fragments in registers: products from buffer cur, step kt + 2 split into the third buffer, step kt + 4 loaded
  auto step = [&](int kt, auto set_t) {
    constexpr int set = decltype(set_t)::value;
    char* nxt = cur + BUF == lds + 3 * BUF ? lds : cur + BUF;
    char* far = nxt + BUF == lds + 3 * BUF ? lds : nxt + BUF;
    meet();
    each<S>([&](auto n_) {
      constexpr int n = decltype(n_)::value, i = n / (6 * NI), at = n % (6 * NI);
      product(set_t, n_);
      if constexpr (i + 1 < MI && at < 3) read_a((set * MI + i + 1) & 1, cur, i + 1, at);
      if constexpr (i + 1 == MI && at < 3 * NI) read_w(set ^ 1, nxt, at);
      if constexpr (i + 1 == MI && at >= 3 * NI && at < 3 * NI + 3) read_a(((set ^ 1) * MI) & 1, nxt, 0, at - 3 * NI);
      constexpr int u0 = first_at(n), u1 = n + 1 == S ? U : first_at(n + 1);
      each<u1 - u0>([&](auto u_) { side(Set<u0 + decltype(u_)::value>{}, set, far, kt + 4); });
      __builtin_amdgcn_sched_barrier(0);
    });
    cur = nxt;
  };
#pragma unroll
  for (int p = 0; p < NP; ++p) load(0, p, 0, 0), load(0, p, 1, 0);
#pragma unroll
  for (int p = 0; p < NP; ++p) load(1, p, 0, 1), load(1, p, 1, 1);
  each<U>([&](auto u_) { side(u_, 0, lds, 2); });
  each<U>([&](auto u_) { side(u_, 1, lds + BUF, 3); });
  meet();
#pragma unroll
  for (int n = 0; n < 3 * NI; ++n) read_w(0, lds, n);
#pragma unroll
  for (int o = 0; o < 3; ++o) read_a(0, lds, 0, o);
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("s_nop 4" ::: "memory");
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    step(kt, Set<0>{});
    step(kt + 1, Set<1>{});
  }
  if (kt < nk) step(kt, Set<0>{});
  if (K % BK) {  // the rest of K, a multiple of 4: elements past the end are zeros
    const int left = K % BK - (tid & 3) * 8;
    meet();
    each<NP>([&](auto p_) {
      constexpr int p = decltype(p_)::value;
      const f32x4_t* a = reinterpret_cast<const f32x4_t*>(src[p] + nk * BK);
      g[0][p][0] = left > 0 ? a[0] : f32x4_t{0.f, 0.f, 0.f, 0.f};
      g[0][p][1] = left > 4 ? a[1] : f32x4_t{0.f, 0.f, 0.f, 0.f};
      each<31>([&](auto q_) { side(Set<p * PER + decltype(q_)::value>{}, 0, lds, 0); });
    });
    meet();
#pragma unroll
    for (int n = 0; n < 3 * NI; ++n) read_w(0, lds, n);
    each<S>([&](auto n_) {
      constexpr int n = decltype(n_)::value;
      if constexpr (n % (6 * NI) == 0) {
#pragma unroll
        for (int o = 0; o < 3; ++o) read_a((n / (6 * NI)) & 1, lds, n / (6 * NI), o);
      }
      product(Set<0>{}, n_);
    });
  }
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");  // the last sums (hipcc does not see into the asm)
  __builtin_amdgcn_sched_barrier(0);

  // rows with a sum that is not finite
  int* marks = reinterpret_cast<int*>(lds + MARK);
  meet();
  if (tid < BM) marks[tid] = 0;
  meet();
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    bool finite = true;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      big[i][j] = big[i][j] + small[i][j];
#pragma unroll
      for (int q = 0; q < 4; ++q) finite &= fabsf(big[i][j][q]) < INFINITY, big[i][j][q] *= SPLIT_DOWN;
    }
    if (!finite) marks[wr * 16 * MI + 16 * i + r16] = 1;
  }
  meet();
  auto out = [&](int r, int c, const f32x4_t& v) {
    if (r >= rows || c >= cols) return;
    float* o = y + (m0 + r) * ldy + n0 + c;
    const float* b = bias + n0 + c;
    if (c + 4 <= cols && (ldy & 3) == 0) {
      f32x4_t s = v;
      if (bias != nullptr) s = s + f32x4_t{b[0], b[1], b[2], b[3]};
      *reinterpret_cast<f32x4_t*>(o) = s;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (c + q < cols) o[q] = v[q] + (bias != nullptr ? b[q] : 0.f);
    }
  };
  const bool any = __any(marks[lane % BM] | marks[(lane + 64) % BM]);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = wr * 16 * MI + 16 * i + r16;
    if (any && marks[r]) continue;
#pragma unroll
    for (int j = 0; j < NI; ++j) out(r, wc * 16 * NI + 16 * j + 4 * kq, big[i][j]);
  }
  if (!any) return;
  MoeTile t;
  t.K = K, t.lds = lds, t.w = reinterpret_cast<const char*>(w + n0 * ldw);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    t.ap[i] = reinterpret_cast<const char*>(x + (m0 + min((tid >> 3) + i * 32, rows - 1)) * ldx) + (tid & 7) * 16;
  moe_tile_many<float, false, 8, 1, 2>(
      t, [&](int j) { return (uint32_t)min(j, cols - 1) * (uint32_t)(ldw * 4); },
      [&](int r, int c, const f32x4_t& v, const f32x4_t&) {
        if (r < BM && marks[r]) out(r, c, v);
      });
}

// y = the ranges' sums in their order (+ bias); N a multiple of 4
__global__ __launch_bounds__(256) void fgemm_reduce_kernel(const float* __restrict__ ws, int ranges, int M, int N,
                                                           const float* __restrict__ bias, float* __restrict__ y, int64_t ldy) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, cols = N / 4;
  if (t >= M * cols) return;
  const int m = (int)(t / cols), n = (int)(t % cols) * 4;
  const float* p = ws + (int64_t)m * N + n;
  f32x4_t s = *reinterpret_cast<const f32x4_t*>(p);
  for (int r = 1; r < ranges; ++r) s = s + *reinterpret_cast<const f32x4_t*>(p + (int64_t)r * M * N);
#pragma unroll
  for (int q = 0; q < 4; ++q) y[m * ldy + n + q] = s[q] + (bias != nullptr ? bias[n + q] : 0.f);
}

// Tiles and their time for a K-step in us, where a CU holds one workgroup and where it holds all it can (measured at M 200 .. 2048).
struct Tile {
  int mi, ni, per_cu;
  double one, full;
};
constexpr Tile TILES[] = {{4, 4, 1, 1.09, 1.19}, {3, 3, 1, 0.77, 0.82}, {4, 2, 1, 0.75, 0.80}, {2, 2, 2, 0.51, 0.81}};

}  // namespace

// The tile for a product of these sizes, as mi * 100 + ni * 10 + ranges of K, or 0: not here. Taken where it is 7 % faster than what the
// vendor's kernels reach (115 TFLOP/s below 2048 rows; 90, seen 65 to 102, where 64 x 64 tiles leave more than a quarter of their second or
// a later round empty: 700 x (2048, 1536) 58 / 42, 700 x (2048, 768) 34 / 25): 350 x (5120, 2048) 65 / 60, not taken; 350 x (11264, 2048) 150 / 111; 350 x (2048,
// 4096) 52 / 64, not taken; from some 500 rows on all of them but narrow ones (700 x (132, 2048) 19 / 33). Ranges of K where
// the tiles leave CUs idle, of at least 16 steps, sums of at most 256 MB: 700 x (2048, 4096) 98 with one, 78 with two.
extern "C" int llmd_fgemm_plan(int M, int N, int K) {
  if (M < 65 || N < 64 || K < 2 * BK || K % 4 || N % 4) return 0;
  double best = 1e30;
  int code = 0;
  const int nk = (K + BK - 1) / BK;
  for (const Tile& t : TILES)
    for (int r = 1; r <= 4; ++r) {
      const int chunk = (K / BK + r - 1) / r;
      const int64_t items = (int64_t)((M + 32 * t.mi - 1) / (32 * t.mi)) * ((N + 32 * t.ni - 1) / (32 * t.ni)) * r;
      if (r > 1 && (chunk < 16 || (r - 1) * chunk >= K / BK || items > 256 || (int64_t)r * M * N > (64 << 20))) continue;
      const int64_t slots = 256 * t.per_cu, last = items % slots;
      const int steps = r > 1 ? chunk : nk;
      double us = 5.0 + (double)(items / slots) * (steps * t.full + 2.0);
      if (last) us += steps * (last <= 256 ? t.one : t.full) + 2.0;
      if (r > 1) us += 5.0 + 1.2e-6 * M * N * r;
      if (us < best) {
        best = us;
        code = t.mi * 100 + t.ni * 10 + r;
      }
    }
  const int64_t blocks = (int64_t)((M + 63) / 64) * ((N + 63) / 64), rounds = (blocks + 255) / 256;
  const double rate = rounds > 1 && 4 * blocks < 3 * 256 * rounds ? 90e6 : 115e6;
  return best < 0.93 * 2.0 * M * N * K / rate + 2.0 ? code : 0;
}

// code: of llmd_fgemm_plan. ws: [ranges, M, N] with more than one range. -1: not taken.
extern "C" int llmd_fgemm(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy, int M, int N, int K,
                          int code, const void* bias, void* ws, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int mi = code / 100, ni = code / 10 % 10, r = code % 10;
  if (K < BK || K % 4 || ldx % 4 || ldw % 4 || (int64_t)TBW * ldw * 4 > 0xffffffffLL) return -1;
  const int chunk = r > 0 ? (K / BK + r - 1) / r : 0;
  if (r < 1 || (r > 1 && (ws == nullptr || N % 4 || (r - 1) * chunk >= K / BK))) return -1;
  const auto launch = [&](auto kernel) {
    const int64_t items = (int64_t)((M + 32 * mi - 1) / (32 * mi)) * ((N + 32 * ni - 1) / (32 * ni)) * r;
    if (items > 0x7fffffff) return -2;
    const bool one = r == 1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)items), dim3(256), 0, st, (const float*)x, ldx, (const float*)w, ldw,
                       one ? (float*)y : (float*)ws, one ? ldy : (int64_t)N, M, N, K, one ? (const float*)bias : nullptr, r);
    if (!one)
      hipLaunchKernelGGL(fgemm_reduce_kernel, dim3((unsigned)(((int64_t)M * (N / 4) + 255) / 256)), dim3(256), 0, st,
                         (const float*)ws, r, M, N, (const float*)bias, (float*)y, ldy);
    return (int)hipGetLastError();
  };
  if (mi == 4 && ni == 4) return launch(fgemm_kernel<4, 4>);
  if (mi == 3 && ni == 3) return launch(fgemm_kernel<3, 3>);
  if (mi == 4 && ni == 2) return launch(fgemm_kernel<4, 2>);
  if (mi == 2 && ni == 2) return launch(fgemm_kernel<2, 2>);
  return -1;
}
