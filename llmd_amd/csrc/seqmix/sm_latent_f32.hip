// Latent attention in fp32 on the matrix cores (v_mfma_f32_16x16x4_f32): absorbed queries [T, H, Dk] over the paged latent cache
// [blocks, bs, Dk], the first R of a row's columns being its values. Dk = 512 or 576, R = 512, pages of whole tiles; other sizes stay
// with the scalar form (sm_latent.hip).
//
// A workgroup takes 16 (token, head) rows and tiles of 32 keys, copied straight to LDS. Scores: wave w takes 16 of the keys and
// half of the columns, S^T = K Q^T, the query in registers; the halves meet in LDS, and every wave makes all of a tile's weights (the lanes of a
// row hold four keys of each block of 16, which is what the second product takes). O^T += V^T P^T: a wave has R / 4 of the
// columns. A row's pieces of 16 bytes lie in the order c ^ (row & 15), so that neither the rows of a key read nor the keys of a value
// read meet in a bank.
// A row's result is the same in every step, whatever else the step holds: the softmax runs over ranges of FR keys at fixed places, joined in
// order; a step of few single tokens deals them to several workgroups, which store them apart, and a second kernel joins them with
// the same operations.
// Bound by the matrix instructions: 136 of 32 cycles per wave and tile, two workgroups per CU. The scalar form has a lane per key, four rows
// per workgroup and no ranges. 16 heads, latent 512 + 64, us, scalar / here: single tokens, two over 75 keys 98 / 19, six over 558 631 / 28, one over
// 4000 6650 / 41; portions, 33 tokens after 73 571 / 22, 173 after 175 1637 / 53, 700 6842 / 166; 64 heads, 300 tokens 5149 / 131.
#include "seqmix_common.h"
#include <algorithm>

using namespace sm;

namespace {

constexpr int NT = 256, KT = 32, FR = 128;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mma(float a, float b, const f32x4_t& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// One more range (m, l): its weight against what is there (mt, lt), which is brought to the new maximum.
__device__ __forceinline__ void join(float& mt, float& lt, float m, float l, float& was, float& now) {
  const float M = fmaxf(mt, m), ref = M == -INFINITY ? 0.f : M;
  was = expf(mt - ref);
  now = expf(m - ref);
  lt = __builtin_fmaf(lt, was, l * now);
  mt = M;
}

// NG: parts of 64 columns of a row; NC: blocks of 16 columns per wave (R = 64 NC). grid: items x groups of 16 heads x range strides.
template <int NG, int NC, bool APART>
__global__ __launch_bounds__(NT, 2) void latent_f32_kernel(
    const float* __restrict__ q_abs, const float* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
    const int* __restrict__ items, const int* __restrict__ row_len, float scale, int H, float* __restrict__ out,
    const float* __restrict__ gate, int64_t gate_stride, int window, float* __restrict__ part_o, float* __restrict__ part_ml, int nsplit) {
  constexpr int Dk = 64 * NG, R = 64 * NC, RB = Dk * 4, PR = Dk / 4, COPIES = KT * PR / NT;
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // the tile, then the scores' halves
  f32x4_t* const half_scores = reinterpret_cast<f32x4_t*>(lds + KT * RB);
  const int item = blockIdx.x, hg = blockIdx.y, G = min(H, 16);
  const int seq = items[item * 3], tok0 = items[item * 3 + 1], ntok = items[item * 3 + 2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  const int myhead = hg * 16 + r16 % G;
  const bool ok = r16 < ntok * G && myhead < H;
  const int mytok = tok0 + (ok ? r16 / G : 0), head = ok ? myhead : hg * 16;
  const int mylen = ok ? row_len[mytok] : 0, mylo = window > 0 ? max(0, mylen - window) : 0;
  const int kend = row_len[tok0 + ntok - 1];
  const int kbase = window > 0 ? max(0, row_len[tok0] - window) / KT * KT : 0;  // the first token has the earliest window
  const int* bt = tables + (int64_t)seq * W;

  const int kb_own = wave & 1, part = wave >> 1;  // of the scores
  f32x4_t qf[2 * NG];
#pragma unroll
  for (int s = 0; s < 2 * NG; ++s)
    qf[s] = *reinterpret_cast<const f32x4_t*>(q_abs + ((int64_t)mytok * H + head) * Dk + 16 * (2 * NG * part + s) + 4 * kq);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 1024;
  const int col0 = wave * 16 * NC;

  float mt = -INFINITY, lt = 0.f;
  f32x4_t ot[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) ot[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int first = kbase / FR, all = (kend - 1) / FR + 1;
  for (int z = blockIdx.z; first + z < all; z += gridDim.z) {
    float m = -INFINITY, l = 0.f;
    f32x4_t o[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int end = min((first + z + 1) * FR, kend);
    for (int k0 = max((first + z) * FR, kbase); k0 < end; k0 += KT) {
      const char* const base = reinterpret_cast<const char*>(cache + ((int64_t)bt[k0 / bs] * bs + k0 % bs) * Dk);
      __syncthreads();  // the tile before is read
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));  // the copies' places are made again for each tile: there are no registers to keep them
#pragma unroll
      for (int i = 0; i < COPIES; ++i) {
        const int e = tid + NT * i, row = e / PR, slot = e - row * PR;
        // keys past the end: the last one again (a page's unwritten rest may hold anything)
        copy_1k(base, (uint32_t)(min(row, kend - 1 - k0) * RB + ((slot & ~15) | ((slot ^ row) & 15)) * 16), lds0 + i * 4096);
      }
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      f32x4_t a4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) a4[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2 * NG; ++s) {
        const int piece = 4 * (2 * NG * part + s) + kq;
        const f32x4_t k = *reinterpret_cast<const f32x4_t*>(lds + (kb_own * 16 + r16) * RB + ((piece & ~15) | ((piece ^ r16) & 15)) * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) a4[j] = mma(k[j], qf[s][j], a4[j]);
      }
      half_scores[(part * 2 + kb_own) * 64 + lane] = (a4[0] + a4[1]) + (a4[2] + a4[3]);
      __syncthreads();
      // this lane's row against keys k0 + 16 kb + 4 kq + r
      float p[2][4], mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const f32x4_t a = half_scores[kb * 64 + lane] + half_scores[(2 + kb) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = k0 + kb * 16 + kq * 4 + r;
          p[kb][r] = (key < mylen) & (key >= mylo) ? a[r] * scale : -INFINITY;
          mx = fmaxf(mx, p[kb][r]);
        }
      }
      mx = row_max(mx);
      const float mn = fmaxf(m, mx), ref = mn == -INFINITY ? 0.f : mn;  // a row with no key yet
      const float corr = expf(m - ref);
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[n][r] *= corr;
      }
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[kb][r] = expf(p[kb][r] - ref);
          sum += p[kb][r];
        }
      l = __builtin_fmaf(l, corr, row_sum(sum));
      m = mn;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 4 * kq + r;
          const char* const v = lds + (kb * 16 + row) * RB + (r16 & 3) * 4;
#pragma unroll
          for (int n = 0; n < NC; ++n) {
            const int piece = (col0 >> 2) + 4 * n + (r16 >> 2);
            o[n] = mma(*reinterpret_cast<const float*>(v + ((piece & ~15) | ((piece ^ row) & 15)) * 16), p[kb][r], o[n]);
          }
        }
    }
    if constexpr (APART) {
      const int64_t at = (((int64_t)item * gridDim.y + hg) * nsplit + z) * 16 + r16;
      if (wave == 0 && kq == 0) {
        part_ml[at * 2] = m;
        part_ml[at * 2 + 1] = l;
      }
#pragma unroll
      for (int n = 0; n < NC; ++n) *reinterpret_cast<f32x4_t*>(part_o + at * R + col0 + 16 * n + 4 * kq) = o[n];
    } else {
      float was, now;
      join(mt, lt, m, l, was, now);
#pragma unroll
      for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) ot[n][r] = __builtin_fmaf(ot[n][r], was, o[n][r] * now);
    }
  }
  if (APART || !ok) return;
  const float inv = 1.f / lt, g = gate ? 1.f / (1.f + expf(-gate[(int64_t)mytok * gate_stride + head])) : 1.f;
  float* dst = out + ((int64_t)mytok * H + head) * R + col0 + 4 * kq;
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    f32x4_t v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = ot[n][r] * inv * g;
    *reinterpret_cast<f32x4_t*>(dst + 16 * n) = v;
  }
}

// Joins the ranges of a step of single tokens (item = token), as the kernel above does.
__global__ __launch_bounds__(NT) void latent_f32_join_kernel(const int* __restrict__ items, const int* __restrict__ row_len, int nsplit,
                                                             const float* __restrict__ part_o, const float* __restrict__ part_ml, int H, int R,
                                                             const float* __restrict__ gate, int64_t gate_stride, float* __restrict__ out, int window) {
  const int item = blockIdx.x, head = blockIdx.y, hg = head >> 4, HG = (H + 15) >> 4;
  const int64_t tok = items[item * 3 + 1];
  const int len = row_len[tok], first = (window > 0 ? max(0, len - window) / KT * KT : 0) / FR;
  const int nz = min((len - 1) / FR + 1 - first, nsplit);
  const int64_t p0 = ((int64_t)item * HG + hg) * nsplit * 16 + (head & 15);
  const float g = gate ? 1.f / (1.f + expf(-gate[tok * gate_stride + head])) : 1.f;
  for (int c = threadIdx.x; c < R; c += NT) {
    float mt = -INFINITY, lt = 0.f, ot = 0.f;
    for (int z = 0; z < nz; ++z) {
      const int64_t p = p0 + (int64_t)z * 16;
      float was, now;
      join(mt, lt, part_ml[p * 2], part_ml[p * 2 + 1], was, now);
      ot = __builtin_fmaf(ot, was, part_o[p * R + c] * now);
    }
    const float inv = 1.f / lt;
    out[(tok * H + head) * R + c] = ot * inv * g;
  }
}

}  // namespace

extern "C" {

int sm_latent_f32_range() { return FR; }

// items: up to 16 / H tokens (one where H > 8) each. nsplit > 1: single tokens, at least as many ranges as any row meets; part_o [items, head groups,
// nsplit, 16, R], part_ml [items, head groups, nsplit, 16, 2]. Returns 0, or 1 when the sizes are outside the compiled forms.
int sm_latent_f32(const void* q_abs, const void* cache, const int* tables, int W, int bs, const int* items, int n_items, const int* row_len,
                  float scale, int H, int R, int Dk, void* out, const void* gate, int64_t gate_stride, int window, int nsplit, float* part_o,
                  float* part_ml, hipStream_t stream) {
  if (R != 512 || (Dk != 512 && Dk != 576) || bs % KT || (((uintptr_t)q_abs | (uintptr_t)cache | (uintptr_t)out) & 15)) return 1;
  if (n_items == 0) return 0;
  const int HG = (H + 15) / 16;
  if (HG > 65535) return 1;
  // about two rounds of workgroups at most: ranges may be planned for contexts far longer than the step's
  const dim3 grid(n_items, HG, std::min(nsplit, std::max(1, 1024 / (HG * n_items))));
  const auto launch = [&](auto kernel) {
    const int lds = KT * Dk * 4 + 4096;
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(kernel, grid, dim3(NT), lds, stream, (const float*)q_abs, (const float*)cache, tables, W, bs, items, row_len, scale, H,
                       (float*)out, (const float*)gate, gate_stride, window, part_o, part_ml, nsplit);
  };
  if (Dk == 576) nsplit > 1 ? launch(latent_f32_kernel<9, 8, true>) : launch(latent_f32_kernel<9, 8, false>);
  else nsplit > 1 ? launch(latent_f32_kernel<8, 8, true>) : launch(latent_f32_kernel<8, 8, false>);
  if (nsplit > 1)
    hipLaunchKernelGGL(latent_f32_join_kernel, dim3(n_items, H), dim3(NT), 0, stream, items, row_len, nsplit, part_o, part_ml, H, R,
                       (const float*)gate, gate_stride, (float*)out, window);
  return 0;
}

}  // extern "C"
