// Shared helpers of the sequence-mixer op library (gfx950 / CDNA4, wave 64).
// Kernels are templated on the activation storage type: float, or bf16 as raw 16-bit words.
// All arithmetic is fp32.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sm {

typedef uint16_t bf16_t;

__device__ __forceinline__ float ld(const float* p) { return *p; }
__device__ __forceinline__ float ld(const bf16_t* p) { return __uint_as_float(((uint32_t)*p) << 16); }
__device__ __forceinline__ void st(float* p, float v) { *p = v; }
__device__ __forceinline__ void st(bf16_t* p, float v) {
  __bf16 h = (__bf16)v;  // round to nearest even
  *p = __builtin_bit_cast(uint16_t, h);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// The larger of a value and those of the lanes 16, 32 and 48 away.
__device__ __forceinline__ float row_max(float v) {
  const uint32_t a = __float_as_uint(v);
  const auto s = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const uint32_t b = __float_as_uint(fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1])));
  const auto t = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}
// The sum of those four values, the same in all of them: (own + 16 away) + (32 away + 48 away).
__device__ __forceinline__ float row_sum(float v) {
  const uint32_t a = __float_as_uint(v);
  const auto s = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const uint32_t b = __float_as_uint(__uint_as_float(s[0]) + __uint_as_float(s[1]));
  const auto t = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

// Wave-wide copy of 1 KB to LDS without registers: lane i's 16 bytes at base + off land at dst + 16 i. Written as asm, so that
// hipcc keeps counting its own LDS reads; the caller waits (vmcnt) before the barrier that publishes the tile.
__device__ __forceinline__ void copy_1k(const char* base, uint32_t off, uint32_t dst) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(off), "s"(base), "s"(__builtin_amdgcn_readfirstlane(dst))
               : "memory");
}

// A projection's output as its product left it: fp32 sums over ranges of K, plane elements apart, added in their order and rounded to
// bf16 as the product's own pass over them does.
struct Parts {
  const float* p;
  int n;
  int64_t plane;
};
template <int W>
__device__ __forceinline__ void add_parts(const Parts& q, int64_t off, float (&v)[W]) {
  static_assert(W % 4 == 0, "");
  const float* p = q.p + off;
  for (int k = 0; k < q.n; k += 4) {  // four loads in flight: one after the other cost 64 rows of 2048 in two streams 3 us of 8
    float4 a[4][W / 4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < W / 4; ++i)
        a[j][i] = *reinterpret_cast<const float4*>(p + (k + j < q.n ? k + j : q.n - 1) * q.plane + 4 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < W / 4; ++i) {
        const float f[4] = {a[j][i].x, a[j][i].y, a[j][i].z, a[j][i].w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k + j < q.n) v[4 * i + e] = k + j == 0 ? f[e] : v[4 * i + e] + f[e];
      }
  }
#pragma unroll
  for (int i = 0; i < W; ++i) v[i] = (float)(__bf16)v[i];
}

// Sum over a workgroup of NT threads (NT a multiple of 64); every thread gets the result.
// The order of the additions is fixed, so a row's result does not depend on the launch.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) s += red[i];
  __syncthreads();
  return s;
}

// Keys per range of a step whose attention rows are cut into ``nsplit`` key ranges. A captured step has as many ranges as the
// longest context it may be replayed with; how many keys they take follows the longest context of the replay (``longest``, on
// the device). ``split_keys`` is the size the ranges were planned with and never exceeded.
// ``least``: keys that a range has at least.
__device__ __forceinline__ int range_keys(const int* longest, int nsplit, int split_keys, int least = 128) {
  if (longest == nullptr) return split_keys;
  const int span = min(*longest, nsplit * split_keys), part = nsplit * 64;
  return min(split_keys, max(least, (span + part - 1) / part * 64));
}
// How many of the ranges can hold keys then: those behind neither run nor are merged. One sequence of 2000 tokens, 16 latent
// heads, ranges planned for 131072: 49.1 us when they did, 20.3 (25.2 planned for 2000).
__device__ __forceinline__ int ranges_used(const int* longest, int nsplit, int split_keys, int least = 128) {
  if (longest == nullptr) return nsplit;
  const int keys = range_keys(longest, nsplit, split_keys, least);
  return max(1, (min(*longest, nsplit * split_keys) + keys - 1) / keys);
}

// One row's results from its key ranges, by a workgroup of NT threads: sum_z b^(m_z - M) o_z / sum_z b^(m_z - M) l_z, M the
// largest m. Range z has (m, l) at ml + z mstep and R numbers at o + z ostep; power(x) = b^x; emit(column, value) is called once
// per column. The ranges' weights are formed once, in LDS; threads take pieces of four columns (R % 4 == 0, else single
// ones) and, as far as there are threads, share the ranges. 16 ranges of 512 columns, 9 rows of 16 heads: 11 us when every
// thread walked all ranges alone and formed the weights again for every column, now 5.1 us. Up to four ranges per row keep that
// walk: a batch of 64 rows of 32 heads, two ranges, 4.6 and 5.2 us with it, 8.3 shared.
template <int NT, typename Power, typename Emit>
__device__ __forceinline__ void merge_ranges(const float* ml, int64_t mstep, const float* o, int64_t ostep, int nsplit, int R,
                                             Power power, Emit emit) {
  constexpr int NZ = 512;
  __shared__ float w[NZ], red[NT / 64];
  __shared__ __attribute__((aligned(16))) float part[NT * 4];
  const int tid = threadIdx.x;
  if (nsplit <= 4) {  // many rows of few ranges (a large batch): nothing to share
    float M = -INFINITY, L = 0.f;
    for (int z = 0; z < nsplit; ++z) M = fmaxf(M, ml[z * mstep]);
    for (int z = 0; z < nsplit; ++z) L += power(ml[z * mstep] - M) * ml[z * mstep + 1];
    for (int c = tid; c < R; c += NT) {
      float a = 0.f;
      for (int z = 0; z < nsplit; ++z) a += power(ml[z * mstep] - M) * o[z * ostep + c];
      emit(c, a / L);
    }
    return;
  }
  float M = -INFINITY;
  for (int z = tid; z < nsplit; z += NT) M = fmaxf(M, ml[z * mstep]);
  M = wave_max(M);
  if ((tid & 63) == 0) red[tid >> 6] = M;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) M = fmaxf(M, red[i]);
  __syncthreads();
  const int cw = R & 3 ? 1 : 4, nc = R / cw;              // columns per piece, pieces
  const int groups = nc < NT ? NT / nc : 1, zg = tid / nc;  // threads that share a piece's ranges
  const int zstep = groups, z_first = groups > 1 ? zg : 0;
  for (int c0 = 0; c0 < nc; c0 += NT) {
    const int c = groups > 1 ? tid - zg * nc : c0 + tid;
    const bool mine = groups > 1 ? zg < groups : c < nc;
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, L = 0.f;
    for (int z0 = 0; z0 < nsplit; z0 += NZ) {
      const int n = min(NZ, nsplit - z0);
      for (int z = tid; z < n; z += NT) {
        w[z] = power(ml[(z0 + z) * mstep] - M);
        L += w[z] * ml[(z0 + z) * mstep + 1];  // an empty range has m = -inf, l = 0
      }
      __syncthreads();
      if (mine) {
        const float* src = o + z0 * ostep + c * cw;
        if (cw == 4) {
#pragma unroll 4
          for (int z = z_first; z < n; z += zstep) {
            const float4 v = *reinterpret_cast<const float4*>(src + z * ostep);
            acc[0] += w[z] * v.x; acc[1] += w[z] * v.y; acc[2] += w[z] * v.z; acc[3] += w[z] * v.w;
          }
        } else {
          for (int z = z_first; z < n; z += zstep) acc[0] += w[z] * src[z * ostep];
        }
      }
      __syncthreads();
    }
    L = block_sum<NT>(L, red);
    if (groups > 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part[tid * 4 + j] = acc[j];
      __syncthreads();
      if (zg == 0)
        for (int i = 1; i < groups; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] += part[(i * nc + c) * 4 + j];
    }
    if (mine && (groups == 1 || zg == 0))
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < cw) emit(c * cw + j, acc[j] / L);
  }
}

// fp32 transcendentals for the sequential scans. float32 storage: the precise library functions.
// bfloat16 storage: the hardware exp2 / log2 / reciprocal forms (about 1 ulp of fp32, far below the
// rounding of the values they are applied to); on a single wave per SIMD the precise forms are most
// of a token's latency.
template <typename T> struct Fn {
  static __device__ __forceinline__ float exp(float x) { return expf(x); }
  static __device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + expf(-x)); }
  static __device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }
  static __device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
  static __device__ __forceinline__ float rsqrt(float x) { return 1.f / sqrtf(x); }
};
template <> struct Fn<uint16_t> {
  static __device__ __forceinline__ float exp(float x) { return __expf(x); }
  static __device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
  static __device__ __forceinline__ float silu(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
  static __device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : __logf(1.f + __expf(x)); }
  static __device__ __forceinline__ float rsqrt(float x) { return __frsqrt_rn(x); }
};

__device__ __forceinline__ float siluf_(float x) { return x / (1.f + expf(-x)); }

// Clamped gated unit: g sigmoid(1.702 g) (v + 1), g cut off above ``limit``, v on both sides.
template <typename T>
__device__ __forceinline__ float clamped_unit(float g, float v, float limit) {
  g = fminf(g, limit);
  v = fminf(fmaxf(v, -limit), limit);
  return g * Fn<T>::sigmoid(1.702f * g) * (v + 1.f);
}

}  // namespace sm
