// Decode GEMM: Y[M, N] = X[M, K] . W[N, K]^T for decode-sized M (1..64), bf16 in,
// fp32 accumulate, bf16 out (SURVEY K08 decode shapes: M = decode batch, N/K of
// the dense projections). At these M the op is a stream over W, so the kernel is
// built around keeping W bytes in flight with NO barrier in the main loop (a
// __syncthreads() fence waits vmcnt(0) and drains the prefetch - the reason the
// round-1 LDS-staged version streamed at 2.4-4 TB/s).
//
// Orientation Y^T = W . X^T on mfma_f32_16x16x32_bf16:
//   A = W rows, 16 B per lane straight from HBM (row r = 16 rb + lane % 16,
//       k = 8 (lane / 16) .. +7 of the current 32-wide k-step);
//   B = X rows, same 16-B fragment shape, straight from L2 (X is re-read by the
//       N / R workgroups of a K range; X/W traffic = M / R).
// Decomposition (host planner `plan`): a workgroup owns R = 16 RB output
// columns (W rows) and one K range of a split-K; its 4 waves split that range
// again in 4 and are summed through LDS at the end (a 2-level tree), so every
// wave streams whole 32-k steps of all RB row blocks. Loads run one chunk of U
// k-steps ahead in two statically indexed register sets.
// Epilogue (act 1: the rows' max(0, .)^2, of the numbers in bf16): bf16 rows when the K range is whole (gridDim.y == 1), else fp32
// partials [split][M][N] summed and rounded by dgemm_reduce_kernel. act 2, whole ranges only: W = [gate; up] of N rows each, a block
// of 16 rows is 8 of gate and the same 8 of up, and silu(gate) * up of the numbers in bf16 is stored. A pass of its own gives the same but where
// the sums, whose order begins elsewhere in K (rot below), fall on the next number in bf16.
//
// NORM: X is rmsnorm(x + res) * gamma, made by every workgroup for itself (the bits of rmsnorm.hip's fused add: the same chunks per
// thread, the same sums) and kept in LDS while its first weights are on their way; the first workgroup stores x + res to res_out, another
// buffer than res, which later workgroups still read. Bound by the weights as without it: what it saves is the norm's launch.
// us of norm, product and (28672) SiLU in a row, apart / here: one row (6144, 4096) 15.9 / 14.7, (28672, 4096) 50.5 / 46.0, (2048, 2048)
// 7.4 / 6.2, two rows 16.2 / 16.1, 52.4 / 50.9, 7.5 / 7.3; four rows lost (16.7 / 19.1): their norms are longer than the launch.
#include "llmd_common.h"

using namespace llmd;

namespace {

constexpr int NT = 256;

struct Norm {
  const uint16_t* x;
  int64_t xs;
  const uint16_t* res;
  int64_t rs;
  const uint16_t* gamma;
  float eps;
  uint16_t* res_out;
  int64_t ros;
};

constexpr int NORM_K = 8192;      // row width of the NORM form
constexpr int NORM_ROWS = 2;      // and its rows

template <int RB, int MB, int U, int OCC, bool NORM>
__device__ __forceinline__ void dgemm(const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ wt,
                                      int64_t w_stride, int M, int N, int K, int nquad_split, uint16_t* __restrict__ y,
                                      int64_t y_stride, float* __restrict__ part, int act, const Norm& norm) {
  __shared__ __attribute__((aligned(16))) f32x4_t red[2][RB][MB][64];
  extern __shared__ __attribute__((aligned(16))) uint16_t xrow[];  // NORM: [M][K]
  __shared__ float ssum[NORM ? NT / 64 : 1];
  const int tile = blockIdx.x, sp = blockIdx.y, nsplit = gridDim.y;
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int row0 = tile * (16 * RB);
  // k range: split sp owns 256-wide blocks [q0, q1); wave wv streams its own
  // contiguous quarter of them in 64-wide steps. A step is two MFMA k-steps
  // whose two 16-B loads per lane cover both halves of one 128-B line of each
  // W row, back to back from one wave (no line shared between waves).
  const int nq = K >> 8;
  const int q0 = sp * nquad_split, q1 = min(nq, q0 + nquad_split);
  const int nqs = max(0, q1 - q0);  // 256-wide blocks in this split = 64-wide steps per wave
  const int nsteps = nqs;
  const int kbase = q0 * 256 + wv * nqs * 64 + 8 * g;

  const uint16_t* wp[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int o = min(row0 / 2 + 8 * rb + (c16 & 7), N - 1);
    const int r = act == 2 ? (c16 < 8 ? o : N + o) : min(row0 + 16 * rb + c16, N - 1);
    wp[rb] = wt + (int64_t)r * w_stride + kbase;
  }
  const uint16_t* xp[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = min(16 * mb + c16, M - 1);
    xp[mb] = NORM ? nullptr : x + (int64_t)m * x_stride + kbase;
  }

  f32x4_t acc[RB][MB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[rb][mb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  u32x4_t wa[U][2][RB], xa[U][2][MB], wb[U][2][RB], xb[U][2][MB];
  // chunk = U steps starting at step s; a step past the end re-reads step 0
  // (valid memory, result unused). No branch may split the main loop: the
  // waitcnt pass then counts loads across blocks conservatively and waits for
  // the prefetched chunk as well.
  // each tile starts its sweep at a rotated step, so concurrent workgroups do
  // not all read the same k column of W (+3-19 % on the 70B shapes, a
  // power-of-two row pitch otherwise piles them onto the same DRAM channels)
  // (act 2: the two workgroups of 16 neighbouring rows of gate alike; apart, (28672, 4096) takes 46.5 us in place of 42.9)
  const int rot = ((act == 2 ? tile >> 1 : tile) * 5) % max(1, nsteps);
  const uint16_t* xl = xrow + min(c16, M - 1) * K + kbase;
  auto load = [&](int s, u32x4_t (&w_)[U][2][RB], u32x4_t (&x_)[U][2][MB], bool with_w = true, bool with_x = true) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int st = s + u < nsteps ? s + u : 0;
      st = st + rot < nsteps ? st + rot : st + rot - nsteps;
      const int64_t off = (int64_t)st * 64;
      if (with_w) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)  // (nontemporal W loads measured 10-30 % slower)
            w_[u][h][rb] = *reinterpret_cast<const u32x4_t*>(wp[rb] + off + 32 * h);
      }
      if (with_x) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            x_[u][h][mb] = *reinterpret_cast<const u32x4_t*>((NORM ? xl : xp[mb]) + off + 32 * h);
      }
    }
  };
  auto mfma_step = [&](const u32x4_t (&w_)[2][RB], const u32x4_t (&x_)[2][MB]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const bf16x8_t af = __builtin_bit_cast(bf16x8_t, w_[h][rb]);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[rb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, __builtin_bit_cast(bf16x8_t, x_[h][mb]),
                                                                acc[rb][mb], 0, 0, 0);
      }
  };
  auto compute = [&](const u32x4_t (&w_)[U][2][RB], const u32x4_t (&x_)[U][2][MB]) {
#pragma unroll
    for (int u = 0; u < U; ++u) mfma_step(w_[u], x_[u]);
  };

  // main loop: pairs of chunks, one chunk always in flight behind the one in use.
  // sched_barrier(0) pins the group order: left alone the scheduler sinks the
  // prefetch loads in between the MFMAs that need the previous chunk, and the
  // counted waits then cover the prefetch too.
  const int npair = nsteps / (2 * U);
  int s = 0;
  if constexpr (NORM) {
    constexpr int VPT = NORM_K / (8 * NT);
    const int nchunk = K >> 3;
    for (int m = 0; m < M; ++m) {
      u32x4_t a[VPT], r[VPT];
#pragma unroll
      for (int c = 0; c < VPT; ++c) {
        const int ci = threadIdx.x + c * NT;
        if (ci < nchunk) {
          a[c] = *reinterpret_cast<const u32x4_t*>(norm.x + m * norm.xs + ci * 8);
          r[c] = *reinterpret_cast<const u32x4_t*>(norm.res + m * norm.rs + ci * 8);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (m == 0 && npair > 0) load(0, wa, xa, true, false);
      __builtin_amdgcn_sched_barrier(0);
      float v[VPT][8], ss = 0.f;
#pragma unroll
      for (int c = 0; c < VPT; ++c) {
        const int ci = threadIdx.x + c * NT;
        if (ci < nchunk) {
          float f[8];
          unpack8(a[c], v[c]);
          unpack8(r[c], f);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] += f[j];
          r[c] = pack8(v[c]);
          unpack8(r[c], v[c]);
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += v[c][j] * v[c][j];
        }
      }
      // barriers that leave the weights in flight
      ss = wave_sum(ss);
      if (lane == 0) ssum[wv] = ss;
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      ss = 0.f;
#pragma unroll
      for (int i = 0; i < NT / 64; ++i) ss += ssum[i];
      const float inv = rsqrtf(ss / (float)K + norm.eps);
#pragma unroll
      for (int c = 0; c < VPT; ++c) {
        const int ci = threadIdx.x + c * NT;
        if (ci < nchunk) {
          float g8[8], o[8];
          unpack8(*reinterpret_cast<const u32x4_t*>(norm.gamma + ci * 8), g8);
#pragma unroll
          for (int j = 0; j < 8; ++j) o[j] = v[c][j] * inv * g8[j];
          *reinterpret_cast<u32x4_t*>(xrow + m * K + ci * 8) = pack8(o);
          if (tile == 0 && sp == 0) *reinterpret_cast<u32x4_t*>(norm.res_out + m * norm.ros + ci * 8) = r[c];
        }
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (npair > 0) load(0, wa, xa, !NORM);
  for (int p = 0; p < npair; ++p, s += 2 * U) {
    load(s + U, wb, xb);
    __builtin_amdgcn_sched_barrier(0);
    compute(wa, xa);
    __builtin_amdgcn_sched_barrier(0);
    load(s + 2 * U, wa, xa);  // the last pair's prefetch is clamped and wasted
    __builtin_amdgcn_sched_barrier(0);
    compute(wb, xb);
    __builtin_amdgcn_sched_barrier(0);
  }
  // tail: < 2U steps, unpipelined
  for (; s < nsteps; ++s) {
    load(s, wb, xb);
    mfma_step(wb[0], xb[0]);
  }

  // ---- sum the 4 waves: (2,3) -> LDS, (0,1) add; 1 -> LDS, 0 adds
  if (wv >= 2) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) red[wv - 2][rb][mb][lane] = acc[rb][mb];
  }
  __syncthreads();
  if (wv < 2) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[rb][mb] += red[wv][rb][mb][lane];
  }
  __syncthreads();
  if (wv == 1) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) red[0][rb][mb][lane] = acc[rb][mb];
  }
  __syncthreads();
  if (wv != 0) return;
  // acc[rb][mb][i] = Y^T[row0 + 16 rb + 4 g + i][16 mb + c16]
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = 16 * mb + c16;
    if (m >= M) continue;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const f32x4_t v = acc[rb][mb] + red[0][rb][mb][lane];
      if (act == 2) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gt = bf2f(f2bf(v[i])), up = __shfl_xor(gt, 32, 64);
          o[i] = gt / (1.f + __expf(-gt)) * up;
        }
        const int n = row0 / 2 + 8 * rb + 4 * g;
        if (g < 2 && n < N)
          *reinterpret_cast<uint2*>(y + (int64_t)m * y_stride + n) = pack4(f32x4_t{o[0], o[1], o[2], o[3]}, 0);
        continue;
      }
      const int n = row0 + 16 * rb + 4 * g;
      if (n >= N) continue;  // N % 4 == 0 (host check): all 4 in or all out
      if (nsplit == 1) {
        *reinterpret_cast<uint2*>(y + (int64_t)m * y_stride + n) = pack4(v, act);
      } else {
        *reinterpret_cast<f32x4_t*>(part + ((int64_t)sp * M + m) * N + n) = v;
      }
    }
  }
}

template <int RB, int MB, int U, int OCC>
__global__ __launch_bounds__(NT, OCC) void dgemm_kernel(const uint16_t* __restrict__ x, int64_t x_stride,
                                                        const uint16_t* __restrict__ wt, int64_t w_stride,
                                                        int M, int N, int K, int nquad_split,
                                                        uint16_t* __restrict__ y, int64_t y_stride,
                                                        float* __restrict__ part, int act) {
  dgemm<RB, MB, U, OCC, false>(x, x_stride, wt, w_stride, M, N, K, nquad_split, y, y_stride, part, act, Norm{});
}

template <int RB, int U, int OCC>
__global__ __launch_bounds__(NT, OCC) void dgemm_norm_kernel(Norm norm, const uint16_t* __restrict__ wt, int64_t w_stride,
                                                             int M, int N, int K, uint16_t* __restrict__ y,
                                                             int64_t y_stride, int act) {
  dgemm<RB, 1, U, OCC, true>(nullptr, 0, wt, w_stride, M, N, K, K >> 8, y, y_stride, nullptr, act, norm);
}

__global__ __launch_bounds__(256) void dgemm_reduce_kernel(const float* __restrict__ part, int nsplit, int M, int N,
                                                           uint16_t* __restrict__ y, int64_t y_stride, int relu2) {
  const int64_t i4 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t total = (int64_t)M * N;
  if (i4 >= total) return;
  const int m = (int)(i4 / N), n = (int)(i4 % N);  // N % 4 == 0: the 4 stay in one row
  f32x4_t s = *reinterpret_cast<const f32x4_t*>(part + i4);
  for (int k = 1; k < nsplit; ++k) s += *reinterpret_cast<const f32x4_t*>(part + (int64_t)k * total + i4);
  *reinterpret_cast<uint2*>(y + (int64_t)m * y_stride + n) = pack4(s, relu2);
}

// register budget per lane: the two chunk sets (2 U steps x 2 loads x (RB + MB)
// x 4) and the row pointers live in arch VGPRs (<= 256); the accumulators
// (4 RB MB) share them at two workgroups per CU, or sit in AGPRs at one
constexpr int vregs(int rb, int mb, int u) { return 16 * u * (rb + mb) + 2 * (rb + mb) + 24; }
constexpr bool fits(int rb, int mb, int u, int occ) {
  return occ == 2 ? vregs(rb, mb, u) + 4 * rb * mb <= 256 : (vregs(rb, mb, u) <= 256 && 4 * rb * mb <= 256);
}
constexpr int pick_u(int rb, int mb, int occ) { return fits(rb, mb, 2, occ) ? 2 : (fits(rb, mb, 1, occ) ? 1 : 0); }

typedef void (*kern_t)(const uint16_t*, int64_t, const uint16_t*, int64_t, int, int, int, int, uint16_t*, int64_t,
                       float*, int);

template <int RB, int MB>
kern_t pick(int occ) {
  if (occ == 2) {
    constexpr int u = pick_u(RB, MB, 2);
    if constexpr (u > 0) return dgemm_kernel<RB, MB, u, 2>;
    return nullptr;
  }
  constexpr int u = pick_u(RB, MB, 1);
  if constexpr (u > 0) return dgemm_kernel<RB, MB, u, 1>;
  return nullptr;
}

template <int MB>
kern_t pick_rb(int rb, int occ) {
  switch (rb) {
    case 1: return pick<1, MB>(occ);
    case 2: return pick<2, MB>(occ);
    case 3: return pick<3, MB>(occ);
    case 4: return pick<4, MB>(occ);
    case 5: return pick<5, MB>(occ);
    case 6: return pick<6, MB>(occ);
    case 7: return pick<7, MB>(occ);
    case 8: return pick<8, MB>(occ);
  }
  return nullptr;
}

kern_t pick_all(int MB, int rb, int occ) {
  return MB == 1 ? pick_rb<1>(rb, occ) : MB == 2 ? pick_rb<2>(rb, occ) : MB == 3 ? pick_rb<3>(rb, occ)
                                                                       : pick_rb<4>(rb, occ);
}

}  // namespace

// 1 if (rb, occ) has an instantiation for this M
extern "C" int llmd_dgemm_supported(int M, int rb, int occ) {
  if (M < 1 || M > 64 || rb < 1 || rb > 8 || (occ != 1 && occ != 2)) return 0;
  const int MB = (M + 15) / 16;
  return pick_u(rb, MB, occ) > 0 ? 1 : 0;
}

// Y = X W^T with a planned decomposition: rb row blocks per workgroup, nsplit
// K splits, occ workgroups per CU. part: nsplit * M * N fp32 when nsplit > 1.
// act: 0 none, 1 squared ReLU, 2 SiLU of the first N rows of W times the other N (nsplit 1). y null: the ranges' sums only, [ranges][M][N]
// in part. Returns the number of ranges, or an error < 0
extern "C" int llmd_skinny_gemm(const void* x, int64_t x_stride, const void* w, int64_t w_stride, int M, int N,
                                int K, int rb, int nsplit, int occ, void* y, int64_t y_stride, float* part,
                                int act, hipStream_t st) {
  if (act < 0 || act > 2 || (act == 2 && (nsplit != 1 || N % 8)) || (y == nullptr && nsplit < 2)) return -1;
  if (M < 1 || M > 64 || K % 256 != 0 || N % 4 != 0 || nsplit < 1 || !llmd_dgemm_supported(M, rb, occ)) return -1;
  const int nq = K / 256;
  const int per = (nq + nsplit - 1) / nsplit;
  nsplit = (nq + per - 1) / per;  // no empty splits
  if (y == nullptr && nsplit < 2) return -3;
  const int MB = (M + 15) / 16;
  kern_t k = pick_all(MB, rb, occ);
  if (k == nullptr) return -2;
  const int cols = act == 2 ? 8 * rb : 16 * rb;
  dim3 grid((N + cols - 1) / cols, nsplit);
  hipLaunchKernelGGL(k, grid, dim3(NT), 0, st, (const uint16_t*)x, x_stride, (const uint16_t*)w, w_stride, M, N, K,
                     per, (uint16_t*)y, y_stride, part, act);
  if (nsplit > 1 && y != nullptr) {
    const int64_t total4 = (int64_t)M * N / 4;
    hipLaunchKernelGGL(dgemm_reduce_kernel, dim3((unsigned)((total4 + 255) / 256)), dim3(256), 0, st, part, nsplit,
                       M, N, (uint16_t*)y, y_stride, act);
  }
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? nsplit : -(int)err;
}

// Y = rmsnorm(x + res, gamma) W^T (act 0) or its SiLU (act 2), res_out = x + res in bf16: the plan's rb and occ, whole K ranges
extern "C" int llmd_skinny_norm(const void* x, int64_t xs, const void* res, int64_t rs, const void* gamma, float eps,
                                void* res_out, int64_t ros, const void* w, int64_t w_stride, int M, int N, int K, int rb,
                                int occ, void* y, int64_t y_stride, int act, hipStream_t st) {
  if (M < 1 || M > NORM_ROWS || K % 256 || K > NORM_K || N % (act == 2 ? 8 : 4) || (act != 0 && act != 2) || xs % 8 || rs % 8 || ros % 8 ||
      res == res_out || !llmd_dgemm_supported(M, rb, occ))
    return -1;
  const Norm norm{(const uint16_t*)x, xs, (const uint16_t*)res, rs, (const uint16_t*)gamma, eps, (uint16_t*)res_out, ros};
  const int cols = act == 2 ? 8 * rb : 16 * rb;
  const dim3 grid((N + cols - 1) / cols);
  const size_t lds = (size_t)M * K * 2;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(NT), lds, st, norm, (const uint16_t*)w, w_stride, M, N, K, (uint16_t*)y, y_stride, act);
    return (int)hipGetLastError();
  };
#define N_CASE(RB)                                                                          \
  if (rb == RB) return occ == 2 ? launch(dgemm_norm_kernel<RB, pick_u(RB, 1, 2), 2>) : launch(dgemm_norm_kernel<RB, pick_u(RB, 1, 1), 1>);
  N_CASE(1) N_CASE(2) N_CASE(3) N_CASE(4) N_CASE(5) N_CASE(6) N_CASE(7) N_CASE(8)
#undef N_CASE
  return -2;
}
