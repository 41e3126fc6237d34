// Dense bf16 GEMM of prompt-sized steps with a tile for every size: C[M, N] = A[M, K] . W[N, K]^T (+ bias), or
// silu(gate) * up of W = [gate; up], or max(0, C)^2. pgemm.hip's 256 x 256 tiles leave CUs idle wherever their number is not a little
// below a multiple of 256; here a tile is 32 MI x 32 NI (64 x 64 .. 256 x 256), chosen so that the tiles fill whole
// rounds of the chip (tgemm_plan below).
//
// What bounds it: large tiles the package power (about 0.95 pJ per operation, 1.5 PFLOP/s); small ones the bytes that a
// CU takes from L2 and reads from LDS per matrix instruction: a K-step of 64 of a 128 x 128 tile needs 512 cycles of the
// matrix units, 512 of the load path (64 B a cycle) and 768 of LDS (32 KB in, 64 KB out, at 128 B) and takes 950.
//
// Four waves of 16 MI x 16 NI, one per SIMD, accumulators in AGPRs. K-steps of 64 stream by LDS-DMA through 2 .. 5 stages
// of LDS (as many as 160 KB hold). A wave reads a step's second half while it multiplies the first, and the next step's
// first half while it multiplies the second. Three stages and more: one barrier per step, behind which the step's stage
// is free and the next one's has landed; two stages (from 192 x 256 on): one barrier for each, half a step apart, so that
// a piece has most of a step to land. Every output is one chain of MFMAs over K in order, whatever the tile: its bits
// do not depend on M (with one range of K).
//
// us, weights cold, hipBLASLt / here: 2048 x (5632, 2048) 51.2 / 40.7, (5120, 2048) 46.2 / 37.2, (2048, 1536) 19.2 / 16.0,
// (2048, 4096) 36.2 / 33.0; 1429 x (4096, 4096) 49.6 / 44.7, (4096, 14336) 152 / 143; 300 x (5120, 2048) 18.3 / 11.9.
// SiLU form, 1429 x (2 x 14336, 4096): 252, with 256 x 256 tiles 280 .. 300.
#include <algorithm>
#include <cmath>

#include "llmd_common.h"

using namespace llmd;

namespace {

constexpr int NT = 256;
constexpr int BK = 64;
constexpr int GROUP_M = 8;   // row tiles that share W's columns in an XCD's run of tiles
constexpr int NUM_CUS = 256;
enum { EPI_NONE = 0, EPI_SILU = 1, EPI_F32 = 2 };

// the accumulator tied to AGPRs: hipcc re-homes loop-carried accumulators of the builtin every iteration
__device__ __forceinline__ void mfma16_acc(f32x4_t& acc, const s16x8_t& a, const s16x8_t& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

__device__ __forceinline__ void bar() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

constexpr int stages(int mi, int ni) { return std::max(2, std::min(5, 40 / (mi + ni))); }
constexpr int lds_bytes(int mi, int ni) {  // the stages, afterwards the waves' images of C
  return std::max(stages(mi, ni) * 4096 * (mi + ni), 4 * 16 * mi * (32 * ni + 16));
}

template <int MI, int NI, int EPI>
__global__ __launch_bounds__(NT, 1) void tgemm_kernel(const uint16_t* __restrict__ A, int64_t lda,
                                                      const uint16_t* __restrict__ W, int64_t ldw,
                                                      uint16_t* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                      const uint16_t* __restrict__ bias, int nsplit,
                                                      int form, float limit, float* __restrict__ ws) {
  constexpr int ST = stages(MI, NI), D = MI + NI, R = MI + NI, T = MI * NI;
  constexpr int STG = 4096 * (MI + NI), OPW = 4096 * MI;
  constexpr int BM = 32 * MI, BN = 32 * NI;
  constexpr int TC = EPI == EPI_SILU ? BN / 2 : BN;  // output columns of a tile
  __shared__ __attribute__((aligned(1024))) char lds[lds_bytes(MI, NI)];  // the ONLY LDS object
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + TC - 1) / TC;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int L = EPI == EPI_F32 ? b % (tiles_m * tiles_n) : b, split = EPI == EPI_F32 ? b / (tiles_m * tiles_n) : 0;
  int tm, tn;
  {
    const int per_group = GROUP_M * tiles_n;
    const int g = L / per_group, first_m = g * GROUP_M;
    const int gm = min(tiles_m - first_m, GROUP_M);
    tm = first_m + (L % per_group) % gm;
    tn = (L % per_group) / gm;
  }
  const int m0 = tm * BM, n0 = tn * TC;
  const int chunk = EPI == EPI_F32 ? (K / BK + nsplit - 1) / nsplit : K / BK;
  const int kbeg = split * chunk, nk = min(chunk, K / BK - kbeg);

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 1, wc = w & 1;

  // rows behind M or N have an offset past the buffer: their pieces are zeros
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)(((M - 1) * lda + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)W, 0, (int)(((EPI == EPI_SILU ? 2 * N : N) - 1) * ldw + K) * 2, 0x00020000);
  uint32_t va[8], vw[8];  // byte offsets of the wave's pieces (sized by MI, NI, hipcc's host pass drops the launch stub)
#pragma unroll
  for (int j = 0; j < MI; ++j) {
    const int row = 8 * (MI * w + j) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    va[j] = m0 + row < M ? (uint32_t)(((m0 + row) * lda + c * 8) * 2) : 0x80000000u;
  }
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int row = 8 * (NI * w + j) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    // SiLU: rows of a fragment of 16 are 8 columns of gate, then the same 8 of up
    const int col = EPI == EPI_SILU ? n0 + (row >> 4) * 8 + (row & 7) : n0 + row;
    const int wrow = EPI == EPI_SILU && (row & 8) ? N + col : col;
    vw[j] = col < N ? (uint32_t)((wrow * ldw + c * 8) * 2) : 0x80000000u;
  }
  // piece p of K-step kt: A pieces, then W pieces. Behind the last step its data again, into a stage nobody reads:
  // the waits below count on it
  auto dma = [&](int kt, char* stage, int p) {
    const uint32_t so = (uint32_t)((kbeg + min(kt, nk - 1)) * BK * 2);
    if (p < MI)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(stage + (MI * w + p) * 1024),
                                               16, va[p < MI ? p : 0], so, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rw, (__attribute__((address_space(3))) void*)(stage + OPW + (NI * w + p - MI) * 1024), 16,
          vw[p >= MI ? p - MI : 0], so, 0, 0);
  };

  const int fr = lane & 15, fq = lane >> 4;
  const int rd0 = fr * 128 + ((fq ^ ((fr >> 1) & 7)) * 16);
  const int rd1 = fr * 128 + (((4 + fq) ^ ((fr >> 1) & 7)) * 16);
  const int a_rd = wr * MI * 2048, w_rd = OPW + wc * NI * 2048;

  f32x4_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  s16x8_t fa0[MI], fw0[NI], fa1[MI], fw1[NI];
  // fragment read r of a set: A 0, the W fragments, the other A fragments
  auto read = [&](s16x8_t(&fa)[MI], s16x8_t(&fw)[NI], const char* stage, int rd, int r) {
    if (r == 0) fa[0] = *reinterpret_cast<const s16x8_t*>(stage + a_rd + rd);
    else if (r <= NI) fw[r <= NI && r > 0 ? r - 1 : 0] = *reinterpret_cast<const s16x8_t*>(stage + w_rd + (r - 1) * 2048 + rd);
    else fa[r > NI ? r - NI : 0] = *reinterpret_cast<const s16x8_t*>(stage + a_rd + (r - NI) * 2048 + rd);
  };

#pragma unroll
  for (int s = 0; s < ST; ++s)
#pragma unroll
    for (int p = 0; p < D; ++p) dma(s, lds + s * STG, p);
  wait_vm<(ST - 1) * D>();
  bar();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    read(fa0, fw0, lds, rd0, r);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 4" ::: "memory");  // v_accvgpr_write (zero init) -> MFMA srcC
  __builtin_amdgcn_sched_barrier(0);

  // half 0: barrier after MFMA TA; half 1: next step's reads after MFMA RB, RB + 1, ...
  constexpr int TA = std::max(R - 1, std::min(T - 1, R + (T - R) / 2));
  constexpr int RB = std::max(1, T - R - T / 6);
  constexpr int SL0 = T - 1 - TA, SL = SL0 + RB - (ST == 2 ? 1 : 0);  // slots that carry DMA pieces
  static_assert(RB + R <= T + 1 || T < 2 * R, "");
  char* cur = lds;
  for (int kt = 0; kt < nk; ++kt) {
    char* nxt = cur + STG;
    if (nxt == lds + ST * STG) nxt = lds;
    auto slot = [&](int s) {
#pragma unroll
      for (int p = 0; p < D; ++p)
        if (p * SL / D == s) dma(kt + ST, cur, p);
    };
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int i = t / NI, j = t % NI;
      if (t <= NI) __builtin_amdgcn_s_waitcnt(0xC07F | ((R - 2 < 15 ? R - 2 : 15) << 8));
      mfma16_acc(acc[i][j], fw0[j], fa0[i]);
      if (t < R) read(fa1, fw1, cur, rd1, t);
      if (t == TA) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's reads of the step are done
        if constexpr (ST > 2) wait_vm<(ST - 2) * D>();
        bar();
      }
      if (t > TA) slot(t - TA - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int i = t / NI, j = t % NI;
      mfma16_acc(acc[i][j], fw1[j], fa1[i]);
      slot(SL0 + t);
      if (ST == 2 && t == RB - 1) {
        wait_vm<D>();
        bar();
      }
      if (t >= RB && t < RB + R) read(fa0, fw0, nxt, rd0, t - RB);
      if (t == T - 1) {
#pragma unroll
        for (int r = T - RB; r < R; ++r) read(fa0, fw0, nxt, rd0, r);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
  }
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");  // the last MFMA results (hipcc does not see into the asm)
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  if constexpr (EPI == EPI_F32) {
    // this range's sums, [nsplit][M][N]
    float* out = ws + ((int64_t)split * M + m0 + wr * 16 * MI + fr) * N + n0 + wc * 16 * NI + 4 * fq;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
        if (m0 + wr * 16 * MI + 16 * i + fr < M && n0 + wc * 16 * NI + 16 * j + 4 * fq < N)
          *reinterpret_cast<f32x4_t*>(out + (int64_t)16 * i * N + 16 * j) = acc[i][j];
    return;
  }
  __syncthreads();

  // acc[i][j][e] = C[16 i + fr][16 j + 4 fq + e] of the wave's part; rows of its image padded by 16 bytes
  constexpr int CH = EPI == EPI_SILU ? NI : 2 * NI;  // 16-byte pieces of a row
  constexpr int PITCH = CH * 16 + 16;
  char* img = lds + w * (16 * MI * PITCH);
  if constexpr (EPI != EPI_SILU) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        f32x4_t v = acc[i][j];
        const int n = n0 + wc * 16 * NI + 16 * j + 4 * fq;
        if (bias != nullptr && n < N) {
          const u32x2_t q = *reinterpret_cast<const u32x2_t*>(bias + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += __uint_as_float(e & 1 ? q[e >> 1] & 0xffff0000u : q[e >> 1] << 16);
        }
        *reinterpret_cast<uint2*>(img + (16 * i + fr) * PITCH + 32 * j + 8 * fq) = pack4(v, form);
      }
  } else {
#pragma unroll
    for (int f = 0; f < T; f += 2) {
      // the halves of two fragments: lanes 0..31 take the first one's gate and up, 32..63 the second one's
      const f32x4_t x = acc[f / NI][f % NI], y = f + 1 < T ? acc[(f + 1 < T ? f + 1 : f) / NI][(f + 1 < T ? f + 1 : f) % NI] : x;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[e]), __float_as_uint(y[e]), false, false);
        float g = __uint_as_float(s[0]), u = __uint_as_float(s[1]);
        if (form) g = __uint_as_float((uint32_t)f2bf(g) << 16), u = __uint_as_float((uint32_t)f2bf(u) << 16);
        if (form == 2) {  // the bits of sm_hyper.hip's clamped units
          g = fminf(g, limit);
          u = fminf(fmaxf(u, -limit), limit);
          o[e] = g * __builtin_amdgcn_rcpf(1.f + __expf(-(1.702f * g))) * (u + 1.f);
        } else {
          o[e] = g / (1.f + __expf(-g)) * u;
        }
      }
      u32x2_t p;
      p[0] = (uint32_t)f2bf(o[0]) | ((uint32_t)f2bf(o[1]) << 16);
      p[1] = (uint32_t)f2bf(o[2]) | ((uint32_t)f2bf(o[3]) << 16);
      const int ff = min(f + (lane >> 5), T - 1);
      *reinterpret_cast<u32x2_t*>(img + (16 * (ff / NI) + fr) * PITCH + 16 * (ff % NI) + 8 * (fq & 1)) = p;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_wave_barrier();
  // (a wave reads only what it wrote)
  const int mw = m0 + wr * 16 * MI, nw = n0 + wc * 8 * CH;
#pragma unroll 4
  for (int q = lane; q < 16 * MI * CH; q += 64) {
    const int row = q / CH, c = q % CH;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(img + row * PITCH + c * 16);
    if (mw + row < M && nw + 8 * c < N) *reinterpret_cast<u32x4_t*>(C + (int64_t)(mw + row) * ldc + nw + 8 * c) = v;
  }
}

// C = the ranges' sums in their order; a thread per 8 columns of a row
__global__ __launch_bounds__(256) void tgemm_reduce_kernel(const float* __restrict__ ws, int nsplit, int M, int N,
                                                           const uint16_t* __restrict__ bias,
                                                           uint16_t* __restrict__ C, int64_t ldc, int relu2) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, cols = N / 8;
  if (t >= M * cols) return;
  const int m = (int)(t / cols), n = (int)(t % cols) * 8;
  const float* p = ws + (int64_t)m * N + n;
  float f[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int s = 0; s < nsplit; ++s, p += (int64_t)M * N) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] += a[e];
      f[4 + e] += b[e];
    }
  }
  if (bias != nullptr) {
    float g[8];
    unpack8(*reinterpret_cast<const u32x4_t*>(bias + n), g);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] += g[e];
  }
  if (relu2) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = relu2_bf(f[e]);
  }
  *reinterpret_cast<u32x4_t*>(C + m * ldc + n) = pack8(f);
}

#define TGEMM_TILES(X)                                                                                           \
  X(2, 2) X(3, 2) X(3, 3) X(3, 4) X(4, 3) X(4, 4) X(4, 6) X(4, 8) X(5, 4) X(5, 6) X(5, 8) X(6, 4) X(6, 6) X(6, 8) \
  X(8, 5) X(8, 6) X(8, 7)

#define T_TILE(MI, NI) {MI, NI},
constexpr int TILES[][2] = {TGEMM_TILES(T_TILE){8, 8}};  // (the last one only with several ranges of K)
#undef T_TILE

// Time of a product in us, fitted to 4305 timings (21 sizes of W, M 65 .. 4500, 18 tiles, one and more ranges of K; off by 6 %; the tile it
// picks is 0.9 % slower than the best one on average; of 2484 random sizes of 21 us and more nine in ten take 3 % less to 21 % more):
// a round is its tiles' fixed part and its K-steps, each bound by the CU (cu: LDS and load path) together with the chip (chip: power and
// L2); the weights' bytes from HBM beside it.
double tgemm_us(int M, int N, int K, int mi, int ni, int ns) {
  const int64_t nt = (int64_t)((M + 32 * mi - 1) / (32 * mi)) * ((N + 32 * ni - 1) / (32 * ni)) * ns;
  const int steps = (K / BK + ns - 1) / ns;
  const double cu = 0.0496 * (mi + ni), chip = 0.01395 * mi * ni + 0.01096 * (mi + ni), one = 0.064 + 0.1496 * mi * ni;
  auto round = [&](double share) { return one + steps * std::sqrt(cu * cu + chip * chip * share * share); };
  double t = (double)(nt / NUM_CUS) * round(1.0);
  if (nt % NUM_CUS) t += round((double)(nt % NUM_CUS) / NUM_CUS);
  const double w = (double)N * K * 2e-6 / 6.6;
  t = 1.95 + std::sqrt(t * t + w * w);
  if (ns > 1) t += 4.69 + 0.643e-6 * M * N * ns;  // the sums and their own launch
  return t;
}

// Whole products on which hipBLASLt is the faster one:
//  * 113 to 128 rows on tiles for two thirds of the CUs, products that wait for their weights: its own 128 rows are split over K, 128 x (15168,
//    6400) 50.3 / 64.7 (105 x (14144, 4288) 43.2 / 39.5, 172 x (19200, 2048) 31.5 / 31.3);
//  * columns in whole tiles of 256, K up to 1024, and 256 x 256 tiles whose rounds the outputs fill by more than 0.8: it overlaps a round's
//    fixed part with the next one, 1920 x (28928, 576) 75.6 / 94.2 (K 1024 to 3072 as full: 1.05 times its time on average).
// 2484 random sizes of 21 us and more (M 65 .. 8192, N 64 .. 32768, K 256 .. 16384, half of each on whole tiles; weights from memory, 25 ms of
// each product at a time: after a pause the clock tells more than the kernel), the library's time over the one here: 1.22 on average, below
// 0.95 in 4.2 % of them, below 0.90 in 1.3 %. On these 2 % it is 0.94; of the others 3.3 % are below 0.95 and 0.5 % below 0.90, the lowest 0.87.
// Below 21 us 0.3 % of 40000 sizes are more than 3 % slower here.
bool left_to_library(int M, int N, int K, int mi, int ni, double us) {
  const int64_t tiles = (int64_t)((M + 32 * mi - 1) / (32 * mi)) * ((N + 32 * ni - 1) / (32 * ni));
  if (us > 21 && M > 112 && M <= 128 && 3 * tiles <= 2 * NUM_CUS) return true;
  const int64_t big = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
  return us > 21 && N % 256 == 0 && K <= 1024 && (double)M * N > 0.8 * (double)((big + 255) / 256 * 256 * 65536);
}

}  // namespace

// The tile for a product of these sizes, as mi * 100 + ni * 10 + ranges of K, or 0: not here. N: rows of W (with silu
// those of gate and up).
//  * Below 65 rows the decode kernels.
//  * Whole products with 256 x 256 tiles and, up to K 2048, those of 256 x 224: pgemm.hip or hipBLASLt as before (2551 x (5632, 2048): hipBLASLt
//    47.5, here 50.6; 2048 x (8192, 8192) 180 both), and those that left_to_library has.
//  * silu 1: in place of the 256 x 256 tiles of pgemm.hip where these take more than 3 % longer (1429 x (28672, 4096) 300 / 252,
//    2048: 359 / 352; 2300: 399 / 399, not taken). silu 2: in place of a product and the activation's own pass, where no
//    more than 5 % slower than 256 x 256 tiles, and only where that product itself has one range of K: 512 x (512, 8192) in two ranges with the
//    activation behind it 18 us, here 26; 300 x (1024, 8192) 23 / 28; of 3500 such sizes the two were 24 % faster on average. Both above mgemm.hip's 256 rows (100 x (28672, 4096): 51, here 53).
//  * More than one range of K only for what the chip takes at once, ranges of at least 8 steps, and where it gains 10 %: 512 x (4096,
//    14336) 98 with one, 65 with four. Sums of at most 256 MB.
extern "C" int llmd_tgemm_plan(int M, int N, int K, int silu) {
  if (M < (silu ? 257 : 65) || N < 8 || K < BK || K % BK) return 0;
  if (silu == 2 && llmd_tgemm_plan(M, N, K, 0) % 10 > 1) return 0;
  double best = 1e30;
  int code = 0, area = 0;
  const int nk = K / BK;
  for (const auto& t : TILES) {
    const int mi = t[0], ni = t[1];
    const int64_t nt = (int64_t)((M + 32 * mi - 1) / (32 * mi)) * ((N + 32 * ni - 1) / (32 * ni));
    for (int ns = 1; ns <= (silu ? 1 : 8); ++ns) {
      const int chunk = (nk + ns - 1) / ns;
      if (ns > 1 && (nt * ns > NUM_CUS || chunk < 8 || (ns - 1) * chunk >= nk || (int64_t)ns * M * N > (64 << 20))) continue;
      const double us = tgemm_us(M, N, K, mi, ni, ns) * (ns > 1 ? 1.1 : 1.0);
      if (us < best) {
        best = us;
        code = mi * 100 + ni * 10 + ns;
        area = mi * ni;
      }
    }
  }
  if (code % 10 == 1 && (area >= 64 || (!silu && ((K <= 2048 && area >= 56) || left_to_library(M, N, K, code / 100, code / 10 % 10, best)))))
    return 0;
  if (silu && best > (silu == 1 ? 0.97 : 1.05) * tgemm_us(M, N, K, 8, 8, 1)) return 0;
  return code;
}

// A tile of llmd_tgemm_plan. N: columns of C; W [N, K], with act 1, 2 and 4 [2 N, K]. act 0: none, 1: silu of gate (the first N rows of W)
// times up (the others), 2: the same of the sums rounded to bf16, as a pass of its own would find them, 3: max(0, .)^2 of the sums rounded
// to bf16, 4: the clamped units g sigmoid(1.702 g) (u + 1), g <= limit and |u| <= limit, of these. bias: [N] or null (no silu).
// Ranges > 1 (no silu): sums in ws [ranges, M, N]. -1: not taken.
extern "C" int llmd_tgemm(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, int M, int N,
                          int K, int act, float limit, int code, const void* bias, void* ws, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int mi = code / 100, ni = code / 10 % 10, nsplit = code % 10;
  if (N % 8 || K % BK || K <= 0 || lda % 8 || ldw % 8 || ldc % 8 || act < 0 || act > 4) return -1;
  const bool silu = act == 1 || act == 2 || act == 4;
  const int nk = K / BK;
  if (nsplit < 1 || nsplit > nk || (nsplit - 1) * ((nk + nsplit - 1) / nsplit) >= nk) return -1;
  if ((nsplit > 1 && (silu || ws == nullptr)) || (bias != nullptr && silu)) return -1;
  // buffer offsets are 31-bit byte offsets
  const int64_t wrows = silu ? 2 * (int64_t)N : N;
  if (((int64_t)(M - 1) * lda + K) * 2 > 0x7fffffffLL || ((wrows - 1) * ldw + K) * 2 > 0x7fffffffLL) return -2;
  const int tc = silu ? 16 * ni : 32 * ni;
  const auto launch = [&](auto kernel) {
    const int64_t grid = (int64_t)((M + 32 * mi - 1) / (32 * mi)) * ((N + tc - 1) / tc) * nsplit;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(NT), 0, st, (const uint16_t*)A, lda, (const uint16_t*)W, ldw,
                       (uint16_t*)C, ldc, M, N, K, (const uint16_t*)bias, nsplit, act == 4 ? 2 : act >= 2, limit, (float*)ws);
    if (nsplit > 1)
      hipLaunchKernelGGL(tgemm_reduce_kernel, dim3((unsigned)(((int64_t)M * (N / 8) + 255) / 256)), dim3(256), 0, st,
                         (const float*)ws, nsplit, M, N, (const uint16_t*)bias, (uint16_t*)C, ldc, act == 3);
    return (int)hipGetLastError();
  };
#define T_CASE(MI, NI)                                                              \
  if (mi == MI && ni == NI)                                                         \
    return silu         ? launch(tgemm_kernel<MI, NI, EPI_SILU>)                    \
           : nsplit > 1 ? launch(tgemm_kernel<MI, NI, EPI_F32>)                     \
                        : launch(tgemm_kernel<MI, NI, EPI_NONE>);
  TGEMM_TILES(T_CASE)
#undef T_CASE
  if (mi == 8 && ni == 8 && nsplit > 1) return launch(tgemm_kernel<8, 8, EPI_F32>);
  return -1;
}
