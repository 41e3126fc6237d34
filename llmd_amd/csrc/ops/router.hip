// Router products: y = x W^T (+ bias) of bf16 rows x [M, K] and weights W [N, K], N small, summed in fp32 and stored as it is or in bf16.
//
// A workgroup's four waves each walk every fourth 64 k of K alone: copies to a ring in LDS of their own (whole 128-byte lines; a fragment
// read from memory straight into registers touches 16 rows and took three times as long), 16 x 16 x 32 matrix instructions, no barrier
// until the four sums of each number are added up, in the waves' order. That order is the same for every size, so a row's numbers
// do not depend on how many rows a step has.
// Bound by the copies into one CU, 24 cycles per KB: (MB + NB) * K * 32 bytes a workgroup, whence the rule in plan() below.
// us over and over, operands in the caches (in a prompt's step of 2048 behind the kernels before it 8.5 in fp32, 7.5 in bf16; of 64 rows
// 4.9); 64 / 1000 / 2048 / 8192 rows; fp32 against the float product of widened copies that stood in its place, and the form of few rows
// (sm_moe.hip router_kernel): (132, 2048) 10.8, 7.2 / 20.8 / 30.8 / 58 -> 3.3 / 5.1 / 6.4 / 15; (256, 7168) 19 / 44 / 71 / 256 -> 7.1 / 13 / 22 /
// 90. Off 64 bits, rms over sums of variance 1: 1.7e-7, 3.9e-7 (long sums of 2048 rows) -> 1.3e-7; K 7168 3.6e-7, 8.7e-7 -> 2.5e-7.
// bf16 against the library / tgemm: (128, 2048) 64 rows 5.5 -> 3.3, 1000 8.3 / 8.8 -> 5.2, 2048 8.8 / 9.1 -> 5.7.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "llmd_common.h"

using namespace llmd;

namespace {

constexpr int NW = 4, NUM_CUS = 256;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int N>
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// D: 64-k steps that a wave's ring holds. nb: blocks of 16 NB columns
template <int MB, int NB, int D, typename Out>
__global__ __launch_bounds__(64 * NW) void router_product_kernel(const uint16_t* __restrict__ x, int64_t xs, const uint16_t* __restrict__ w,
                                                                 int64_t ws, int M, int N, int K, int nb,
                                                                 const uint16_t* __restrict__ bias, Out* __restrict__ y) {
  constexpr int R = MB + NB, STEP = R * 2048;
  static_assert(MB * NB * NW * 1024 <= NW * D * STEP && (D - 1) * 2 * R < 64, "");
  __shared__ __attribute__((aligned(1024))) char ring[NW * D * STEP];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  // an XCD takes whole groups of rows: its L2 reads them once for all their blocks of columns
  const int at = blockIdx.x >> 3, m0 = (at / nb * 8 + (blockIdx.x & 7)) * 16 * MB, n0 = at % nb * 16 * NB;
  if (m0 >= M) return;
  char* mine = ring + wave * (D * STEP);
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_addr(mine));
  // copy j of a step brings eight rows of 128 bytes; a 16-byte piece's place in its row is turned by the row's number, which
  // gives the lanes of a read banks of their own
  const char* from[2 * R];
#pragma unroll
  for (int j = 0; j < 2 * R; ++j) {
    const int row = 8 * j + (lane >> 3), piece = ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    from[j] = j < 2 * MB ? (const char*)(x + min(m0 + row, M - 1) * xs) + piece : (const char*)(w + min(n0 + row - 16 * MB, N - 1) * ws) + piece;
  }
  const auto fetch = [&](int step, int slot) {
#pragma unroll
    for (int j = 0; j < 2 * R; ++j) glds16(from[j] + (int64_t)step * 128, lds + slot * STEP + j * 1024);
  };
  f32x4_t acc[MB][NB] = {};
  const int steps = K / 64;
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (wave + NW * d < steps) fetch(wave + NW * d, d);
  int slot = 0;
  for (int s = wave; s < steps; s += NW) {
    if (s + NW * (D - 1) < steps) {
      fetch(s + NW * (D - 1), slot == 0 ? D - 1 : slot - 1);
      wait_copies<(D - 1) * 2 * R>();
    } else {
      wait_copies<0>();
    }
    const char* t = mine + slot * STEP;
    slot = slot + 1 == D ? 0 : slot + 1;
    bf16x8_t f[2][R];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < R; ++i)
        f[h][i] = *reinterpret_cast<const bf16x8_t*>(t + (16 * i + r16) * 128 + ((4 * h + g) ^ ((r16 >> 1) & 7)) * 16);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[h][MB + j], f[h][i], acc[i][j], 0, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is read before it is filled again
  }
  __syncthreads();
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(ring);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) sums[(wave * MB * NB + i * NB + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int t = wave; t < MB * NB; t += NW) {
    f32x4_t v = sums[t * 64 + lane];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += sums[(i * MB * NB + t) * 64 + lane];
    // v[r] = y[m][n + r]
    const int m = m0 + t / NB * 16 + r16, n = n0 + t % NB * 16 + 4 * g;
    if (m >= M) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) {
        const float s = bias ? v[r] + bf2f(bias[n + r]) : v[r];
        if constexpr (sizeof(Out) == 4) y[(int64_t)m * N + n + r] = s;
        else y[(int64_t)m * N + n + r] = f2bf(s);
      }
  }
}

// Rows and columns of a workgroup in blocks of 16, by what the fullest CU copies: its workgroups times MB + NB. us, 16 x 16 / 32 x 32 / 32 x 48 of
// (132, 2048): 64 rows 3.3 / 4.6 / 5.5, 512 4.4 / 4.7 / 5.7, 1000 6.5 / 5.1 / 5.9, 1700 8.5 / 7.4 / 6.1, 2551 11.2 / 8.0 / 6.8, 8192 28 / 17.5 / 15.
constexpr int FORMS[3][2] = {{1, 1}, {2, 2}, {2, 3}};
int plan(int M, int N, int64_t* copies) {
  int form = 0;
  *copies = INT64_MAX;
  for (int i = 0; i < 3; ++i) {
    const int r = 16 * FORMS[i][0], c = 16 * FORMS[i][1];
    const int64_t n = (int64_t)((M + r - 1) / r) * ((N + c - 1) / c), cost = (n + NUM_CUS - 1) / NUM_CUS * (FORMS[i][0] + FORMS[i][1]);
    if (cost < *copies) *copies = cost, form = i;
  }
  return form;
}

}  // namespace

// The form (0 .. 2) for these sizes, -1: the other products are faster. That is never so in fp32; in bf16 it is where a CU has more than
// one of the larger workgroups, or has one that walks long rows: us, here / the better of tgemm and library, 2551 x (128, 2048) 6.7 / 9.2,
// 4096 9.2 / 9.3, 8192 14.7 / 10.4; 512 x (512, 4096) 8.9 / 10.4, 1000 14.2 / 13.5; 200 x (256, 7168) 7.6 / 9.3, 512 12.5 / 11.3.
extern "C" int llmd_router_form(int M, int N, int K, int f32) {
  if (M <= 0 || N <= 0 || K < 64 || K % 64) return -1;
  int64_t copies;
  const int form = plan(M, N, &copies);
  return f32 || copies <= FORMS[0][0] + FORMS[0][1] || (copies <= FORMS[2][0] + FORMS[2][1] && K <= 4096) ? form : -1;
}

// f32: y [M, N] in fp32, else bf16. bias: [N] or null. x rows xs apart, w rows ws: multiples of 8, from 16-byte addresses. form: of
// llmd_router_form. -1: not these sizes
extern "C" int llmd_router_product(const void* x, int64_t xs, const void* w, int64_t ws, int M, int N, int K, const void* bias, int f32,
                                   void* y, int form, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 64 || K % 64 || xs % 8 || ws % 8 || form < 0 || form > 2) return -1;
  const auto go = [&](auto kernel, auto* out) {
    const int mb = FORMS[form][0], cols = 16 * FORMS[form][1], nb = (N + cols - 1) / cols;
    const int64_t grid = ((int64_t)((M + 16 * mb - 1) / (16 * mb)) + 7) / 8 * 8 * nb;
    if (grid > INT32_MAX) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * NW), 0, st, (const uint16_t*)x, xs, (const uint16_t*)w, ws, M, N, K, nb,
                       (const uint16_t*)bias, out);
    return (int)hipGetLastError();
  };
#define R_GO(MB, NB, D) \
  return f32 ? go(router_product_kernel<MB, NB, D, float>, (float*)y) : go(router_product_kernel<MB, NB, D, uint16_t>, (uint16_t*)y)
  if (form == 0) R_GO(1, 1, 4);
  if (form == 1) R_GO(2, 2, 2);
  R_GO(2, 3, 2);
#undef R_GO
}
