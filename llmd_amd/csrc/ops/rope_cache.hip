// Fused rotary embedding + paged KV-cache write (vLLM
// `rotary_embedding` + `reshape_and_cache` fused into one pass).
//
// Input is the raw output of the fused QKV projection, qkv[T, (Hq+2Hkv)*D].
//   * Q heads are rotated in place (the attention kernels read Q through a row stride).
//   * K heads are rotated and scattered into the paged cache at slot_mapping[t].
//   * V heads are copied into the paged cache.
// Paged cache layout (per layer view; see llmd_amd/engine/kv_cache.py):
//   element (block b, kv head h, row r, dim d) at  b*block_stride + h*bs*D + r*D + d
// with the K and V planes given as separate base pointers. A whole block of one
// layer is therefore one contiguous [Hkv, bs, D] slab, which is the unit moved by
// KV transfer (kvx) and offload.
// cos_sin[pos, 0:R/2] = cos, cos_sin[pos, R/2:R] = sin, f32, R = rotary dim.
#include "llmd_common.h"

using namespace llmd;

namespace {

constexpr int NT = 256;

// NEOX = rotate_half pairing (d, d + R/2); otherwise GPT-J interleaved pairs (2i, 2i+1).
// F8: the cache is e4m3fn; K/V are multiplied by kinv/vinv (1/k_scale, 1/v_scale)
// and saturated on the way in (SURVEY K06 "quantize K/V", K16).
// One token row: `src` is the projection output row (global, or an LDS copy), rotated Q goes to
// `row` (the qkv buffer row the attention reads), rotated K and V to the cache. NTH threads.
// ND 64, 128 or 256: heads of that size, all of it rotated in halves, whose RMS norm (qw, kw) comes first, the bits of
// rmsnorm.hip's qk_rmsnorm_kernel: that kernel's lane holds E = ND / 64 neighbours and its sums meet at distances 32, 16 .. 1, so
// here the pairs (d, d + ND / 2) of an item meet first, then the head's other items, then what an item holds. ND 0: no norm.
template <bool NEOX, bool F8, int NTH, int ND = 0>
__device__ __forceinline__ void rope_row(const uint16_t* src, uint16_t* row, int t,
                                         const int64_t* __restrict__ positions, const float* __restrict__ cos_sin,
                                         int rot, int Hq, int Hkv, int D, const int64_t* __restrict__ slots,
                                         void* __restrict__ kc, void* __restrict__ vc, int64_t block_stride, int bs,
                                         float kinv, float vinv, const uint16_t* __restrict__ qw = nullptr,
                                         const uint16_t* __restrict__ kw = nullptr, float eps = 0.f) {
  static_assert(ND == 0 || NEOX, "");
  const int64_t pos = positions[t];
  const float* cs = cos_sin + pos * rot;
  const int64_t slot = slots ? slots[t] : -1;
  LLMD_DCHECK(slot >= -1);  // -1 = padded row (graph buckets), else a cache slot
  int64_t cache_off = -1;
  if (slot >= 0) {
    const int64_t blk = slot / bs, r = slot % bs;
    cache_off = blk * block_stride + r * D;
  }
  const int half = rot / 2;
  // --- rotation work: (Hq + Hkv) heads x (rot/16) items of 8 pairs
  const int items_per_head = rot / 16;
  const int n_rot = (Hq + Hkv) * items_per_head;
  for (int it = threadIdx.x; it < n_rot; it += NTH) {
    const int h = it / items_per_head, c = it % items_per_head;
    const uint16_t* hp = src + h * D;
    float a[8], b[8], co[8], si[8];
    int ia, ib;  // element offsets of the two 8-wide operands
    if (NEOX) {
      ia = c * 8;
      ib = half + c * 8;
      u32x4_t va = *reinterpret_cast<const u32x4_t*>(hp + ia);
      u32x4_t vb = *reinterpret_cast<const u32x4_t*>(hp + ib);
      unpack8(va, a);
      unpack8(vb, b);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        co[j] = cs[c * 8 + j];
        si[j] = cs[half + c * 8 + j];
      }
    } else {
      // 16 consecutive elements = 8 interleaved pairs
      ia = c * 16;
      ib = c * 16 + 8;
      u32x4_t va = *reinterpret_cast<const u32x4_t*>(hp + ia);
      u32x4_t vb = *reinterpret_cast<const u32x4_t*>(hp + ib);
      float e[16];
      unpack8(va, e);
      unpack8(vb, e + 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        a[j] = e[2 * j];
        b[j] = e[2 * j + 1];
        co[j] = cs[c * 8 + j];
        si[j] = cs[half + c * 8 + j];
      }
    }
    if constexpr (ND != 0) {
      constexpr int E = ND / 64, IT = ND / 16;  // a head's items are IT neighbouring lanes
      float q[8 / E];
#pragma unroll
      for (int l = 0; l < 8 / E; ++l) {
        float p = 0.f, r = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          p += a[l * E + e] * a[l * E + e];
          r += b[l * E + e] * b[l * E + e];
        }
        q[l] = p + r;
      }
#pragma unroll
      for (int o = IT / 2; o > 0; o >>= 1)
#pragma unroll
        for (int l = 0; l < 8 / E; ++l) q[l] += __shfl_xor(q[l], o, 64);
#pragma unroll
      for (int o = 4 / E; o > 0; o >>= 1)
#pragma unroll
        for (int l = 0; l < o; ++l) q[l] += q[l + o];
      const float inv = rsqrtf(q[0] / (float)ND + eps);
      const uint16_t* w = h < Hq ? qw : kw;
      float wa[8], wb[8];
      unpack8(*reinterpret_cast<const u32x4_t*>(w + ia), wa);
      unpack8(*reinterpret_cast<const u32x4_t*>(w + ib), wb);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        wa[j] *= a[j] * inv;
        wb[j] *= b[j] * inv;
      }
      unpack8(pack8(wa), a);
      unpack8(pack8(wb), b);
    }
    float oa[8], ob[8];
    // (fmaf: a contraction left to the compiler is not the same one in each of these kernels. Element 0 is as it was before they were
    // written out, so that the bits stay)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      oa[j] = fmaf(a[j], co[j], -(b[j] * si[j]));
      ob[j] = j ? fmaf(b[j], co[j], a[j] * si[j]) : fmaf(a[j], si[j], b[j] * co[j]);
    }
    u32x4_t pa, pb;
    if (NEOX) {
      pa = pack8(oa);
      pb = pack8(ob);
    } else {
      float e[16];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[2 * j] = oa[j];
        e[2 * j + 1] = ob[j];
      }
      pa = pack8(e);
      pb = pack8(e + 8);
    }
    if (h < Hq) {
      *reinterpret_cast<u32x4_t*>(row + h * D + ia) = pa;
      *reinterpret_cast<u32x4_t*>(row + h * D + ib) = pb;
    } else if (cache_off >= 0) {
      const int64_t dst = cache_off + (int64_t)(h - Hq) * bs * D;
      store8_from_bf16<F8>(kc, dst + ia, pa, kinv);
      store8_from_bf16<F8>(kc, dst + ib, pb, kinv);
    }
  }
  if (cache_off < 0) return;
  // --- K pass-through dims beyond the rotary dim, and V copy
  const int cpr = D / 8;             // 16-B chunks per head
  const int kpass = (D - rot) / 8;   // un-rotated K chunks per head
  const int n_copy = Hkv * (kpass + cpr);
  for (int it = threadIdx.x; it < n_copy; it += NTH) {
    const int per = kpass + cpr;
    const int h = it / per, c = it % per;
    if (c < kpass) {
      const int e = rot + c * 8;
      u32x4_t v = *reinterpret_cast<const u32x4_t*>(src + (Hq + h) * D + e);
      store8_from_bf16<F8>(kc, cache_off + (int64_t)h * bs * D + e, v, kinv);
    } else {
      const int e = (c - kpass) * 8;
      u32x4_t v = *reinterpret_cast<const u32x4_t*>(src + (Hq + Hkv + h) * D + e);
      store8_from_bf16<F8>(vc, cache_off + (int64_t)h * bs * D + e, v, vinv);
    }
  }
}

template <bool NEOX, bool F8, int ND>
__global__ __launch_bounds__(NT) void rope_cache_kernel(
    uint16_t* __restrict__ qkv, int64_t qkv_stride, const int64_t* __restrict__ positions,
    const float* __restrict__ cos_sin, int rot, int Hq, int Hkv, int D,
    const int64_t* __restrict__ slots, void* __restrict__ kc, void* __restrict__ vc,
    int64_t block_stride, int bs, float kinv, float vinv, const uint16_t* __restrict__ qw,
    const uint16_t* __restrict__ kw, float eps) {
  const int t = blockIdx.x;
  uint16_t* row = qkv + (int64_t)t * qkv_stride;
  rope_row<NEOX, F8, NT, ND>(row, row, t, positions, cos_sin, rot, Hq, Hkv, D, slots, kc, vc, block_stride, bs, kinv,
                             vinv, qw, kw, eps);
}

// The decode step's QKV projection split-K partials (fp32 [nsplit][T][W], csrc/ops/mgemm.hip) summed
// and rounded to bf16 exactly as mgemm_reduce_kernel does, staged in LDS (and stored to the qkv row),
// then RoPE + the paged cache write from the LDS copy: one launch instead of reduce + rope_cache,
// bit-identical to them. 1024 threads per token row (the partials stream with enough loads in flight).
constexpr int RNT = 1024;
constexpr int RMAXW = 24576;  // row width (elements) the 48 KB LDS copy holds

template <bool NEOX, bool F8, int ND>
__global__ __launch_bounds__(RNT) void reduce_rope_cache_kernel(
    const float* __restrict__ part, int nsplit, int T, int W, uint16_t* __restrict__ qkv, int64_t qkv_stride,
    const int64_t* __restrict__ positions, const float* __restrict__ cos_sin, int rot, int Hq, int Hkv, int D,
    const int64_t* __restrict__ slots, void* __restrict__ kc, void* __restrict__ vc, int64_t block_stride, int bs,
    float kinv, float vinv, const uint16_t* __restrict__ qw, const uint16_t* __restrict__ kw, float eps) {
  __shared__ __attribute__((aligned(16))) uint16_t lrow[RMAXW];
  const int t = blockIdx.x;
  const int64_t total = (int64_t)T * W;
  uint16_t* row = qkv + (int64_t)t * qkv_stride;
  for (int c = threadIdx.x; c < W / 8; c += RNT) {
    const float* p = part + (int64_t)t * W + c * 8;
    f32x4_t s0 = *reinterpret_cast<const f32x4_t*>(p), s1 = *reinterpret_cast<const f32x4_t*>(p + 4);
    for (int k = 1; k < nsplit; ++k) {
      s0 += *reinterpret_cast<const f32x4_t*>(p + (int64_t)k * total);
      s1 += *reinterpret_cast<const f32x4_t*>(p + (int64_t)k * total + 4);
    }
    const float y[8] = {s0[0], s0[1], s0[2], s0[3], s1[0], s1[1], s1[2], s1[3]};
    const u32x4_t v = pack8(y);
    *reinterpret_cast<u32x4_t*>(lrow + c * 8) = v;
    *reinterpret_cast<u32x4_t*>(row + c * 8) = v;  // the un-rotated projection, as the two-kernel path leaves K / V
  }
  __syncthreads();
  rope_row<NEOX, F8, RNT, ND>(lrow, row, t, positions, cos_sin, rot, Hq, Hkv, D, slots, kc, vc, block_stride, bs, kinv,
                              vinv, qw, kw, eps);
}

// qw, kw (both or neither): the heads' norm weights, for heads of 64, 128 or 256 that neox rotates whole
int norm_size(const void* qw, const void* kw, int D, int rot, int neox) {
  if (qw == nullptr && kw == nullptr) return 0;
  return qw != nullptr && kw != nullptr && neox && rot == D && (D == 64 || D == 128 || D == 256) ? D : -1;
}

#define ROPE_DISPATCH(LAUNCH)                                          \
  if (!neox) {                                                         \
    if (fp8) LAUNCH(false, true, 0); else LAUNCH(false, false, 0);     \
  } else if (nd == 0) {                                                \
    if (fp8) LAUNCH(true, true, 0); else LAUNCH(true, false, 0);       \
  } else if (nd == 64) {                                               \
    if (fp8) LAUNCH(true, true, 64); else LAUNCH(true, false, 64);     \
  } else if (nd == 128) {                                              \
    if (fp8) LAUNCH(true, true, 128); else LAUNCH(true, false, 128);   \
  } else {                                                             \
    if (fp8) LAUNCH(true, true, 256); else LAUNCH(true, false, 256);   \
  }

}  // namespace

extern "C" int llmd_reduce_rope_cache(const float* part, int nsplit, int W, void* qkv, int64_t qkv_stride,
                                      const int64_t* positions, const float* cos_sin, int rot, int Hq, int Hkv,
                                      int D, const int64_t* slots, void* kc, void* vc, int64_t block_stride, int bs,
                                      int T, int neox, int fp8, float kinv, float vinv, const void* qw, const void* kw,
                                      float eps, hipStream_t st) {
  if (T == 0) return 0;
  const int nd = norm_size(qw, kw, D, rot, neox);
  if (W % 8 || W > RMAXW || W < (Hq + 2 * Hkv) * D || qkv_stride % 8 || nsplit < 1 || nd < 0) return -1;
  dim3 g(T), b(RNT);
#define LAUNCH(NX, F8, ND)                                                                                      \
  hipLaunchKernelGGL((reduce_rope_cache_kernel<NX, F8, ND>), g, b, 0, st, part, nsplit, T, W, (uint16_t*)qkv,   \
                     qkv_stride, positions, cos_sin, rot, Hq, Hkv, D, slots, kc, vc, block_stride, bs, kinv, vinv, \
                     (const uint16_t*)qw, (const uint16_t*)kw, eps)
  ROPE_DISPATCH(LAUNCH)
#undef LAUNCH
  return (int)hipGetLastError();
}

// With norm weights in place of rmsnorm.hip's pass (2048 rows of 40 heads of 128: 13.9 + 10.2 us, here 13.3;
// 64 rows 4.8 + 4.9, and 4.7 for the sums over ranges of K that precede them, here 5.1 with these)
extern "C" int llmd_rope_cache(void* qkv, int64_t qkv_stride, const int64_t* positions,
                               const float* cos_sin, int rot, int Hq, int Hkv, int D,
                               const int64_t* slots, void* kc, void* vc, int64_t block_stride,
                               int bs, int T, int neox, int fp8, float kinv, float vinv, const void* qw, const void* kw,
                               float eps, hipStream_t st) {
  if (T == 0) return 0;
  const int nd = norm_size(qw, kw, D, rot, neox);
  if (nd < 0) return -1;
  dim3 g(T), b(NT);
#define LAUNCH(NX, F8, ND)                                                                                \
  hipLaunchKernelGGL((rope_cache_kernel<NX, F8, ND>), g, b, 0, st, (uint16_t*)qkv, qkv_stride, positions, \
                     cos_sin, rot, Hq, Hkv, D, slots, kc, vc, block_stride, bs, kinv, vinv, (const uint16_t*)qw, \
                     (const uint16_t*)kw, eps)
  ROPE_DISPATCH(LAUNCH)
#undef LAUNCH
  return 0;
}
