#pragma once
// The softmax that the attention forms for prompts share (sm_gqa.hip, sm_latent.hip).
#include "seqmix_common.h"

namespace sm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int MKT = 32;  // keys per tile

// Online softmax of 16 rows over tiles of 32 keys, shared by the forms for prompts (a row has the same bits in each). A lane holds one
// row's scores of eight neighbouring keys, 8 kq .. 8 kq + 7 of the tile, which four lanes share.
// The weights are exp2(score - ref), and a row's ref moves only when one of its own scores passes it by 2^RISE: after a row's
// first tiles a step has neither a maximum across lanes nor products with the accumulators. Every row decides for itself (one that
// stays is multiplied by 1), so its bits do not depend on the rows beside it. The sums stay with the lanes until the end.
constexpr float RISE = 8.f;
constexpr float LOW_SINK = -0x1p20f;  // (base 2; above it a reference is off by a sixteenth at most)

// (fmaxf takes an instruction more for each operand)
__device__ __forceinline__ float max3(float a, float b, float c) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

struct RowSoftmax {
  float ref;   // what the weights are relative to; 0 before the first key
  float rise;  // ref moves when a score passes it by more: -infinity before the first key
  float l;     // this lane's part of the sum of weights
  // a sink is a score that is already counted, or one that is counted behind all keys: far below them it would take the digits of the
  // reference that follows it (ref + mx is -1e10 + 1e10), and -infinity has no difference from itself
  __device__ __forceinline__ void start(const float* sinks, int head, int kq) {
    const float sink = sinks ? sinks[head] * 1.44269504088896341f : -INFINITY;
    const bool later = sink <= LOW_SINK;
    ref = later ? 0.f : sink;
    rise = later ? -INFINITY : RISE;
    l = !later && kq == 0 ? 1.f : 0.f;
  }
  template <int NCB>
  __device__ __forceinline__ void finish(const float* sinks, int head, int kq, f32x4_t (&o)[NCB]) {
    asm volatile("" : "+v"(head));  // loaded again: no register is kept for it
    const float sink = sinks ? sinks[head] * 1.44269504088896341f : -INFINITY;
    if (!(sink <= LOW_SINK) || sink == -INFINITY) return;
    const bool above = rise < 0.f || sink > ref;
    const float corr = rise < 0.f || !above ? 1.f : __builtin_amdgcn_exp2f(ref - sink);
#pragma unroll
    for (int n = 0; n < NCB; ++n) o[n] *= corr;
    l = l * corr + (kq > 0 ? 0.f : above ? 1.f : __builtin_amdgcn_exp2f(sink - ref));
    if (above) ref = sink, rise = RISE;
  }
  __device__ __forceinline__ float top() const { return rise < 0.f ? -INFINITY : ref; }
};

// a: the products of this lane's row with keys key0 .. key0 + 7 of a tile (i = 4 kb + r in a[kb][r]); x: what the weights are exp2 of
__device__ __forceinline__ void row_scores(const f32x4_t (&a)[2], float scale2, float slope, bool sloped, int dist, float ref, float (&x)[8]) {
  if (sloped) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(a[i >> 2][i & 3], scale2, __builtin_fmaf(-slope, (float)dist - (float)i, -ref));
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(a[i >> 2][i & 3], scale2, -ref);
  }
}
__device__ __forceinline__ float top8(const float (&x)[8]) {
  return max3(max3(x[0], x[1], x[2]), max3(x[3], x[4], x[5]), max3(x[6], x[7], x[7]));
}
// the weights in two bf16 parts: hi = a weight's upper 16 bits (truncated), lo = the upper 16 bits of the exact rest; hi + lo
// differs from the fp32 weight by less than 2^-16 of it, with no rounding arithmetic
__device__ __forceinline__ void row_weights(const float (&x)[8], RowSoftmax& s, bf16x8_t& pah, bf16x8_t& pal) {
  float p[8];
  u32x4_t hw, lw;
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(x[i]);
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const uint32_t u0 = __float_as_uint(p[i]), u1 = __float_as_uint(p[i + 1]);
    const uint32_t r0 = __float_as_uint(p[i] - __uint_as_float(u0 & 0xffff0000u));
    const uint32_t r1 = __float_as_uint(p[i + 1] - __uint_as_float(u1 & 0xffff0000u));
    hw[i >> 1] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // the upper halves of both
    lw[i >> 1] = __builtin_amdgcn_perm(r1, r0, 0x07060302u);
  }
  pah = __builtin_bit_cast(bf16x8_t, hw);
  pal = __builtin_bit_cast(bf16x8_t, lw);
  s.l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
}
// A tile for one block of rows. From mylen on, outside of its chunk (from mylo) and its window (from mywlo, and below keep) a row
// sees nothing; plain: every row sees the whole tile.
template <int NCB, bool CALM>
__device__ __forceinline__ void weigh(const f32x4_t (&a)[2], float scale2, float slope, bool sloped, bool plain, int key0, int mylen,
                                      int mylo, int mywlo, int keep, RowSoftmax& s, f32x4_t (&o)[NCB], bf16x8_t& pah, bf16x8_t& pal) {
  float x[8];
  if (CALM && plain && !sloped) {  // most tiles: no mask, and no row's reference moves
    row_scores(a, scale2, 0.f, false, 0, s.ref, x);
    if (!__any(top8(x) > s.rise)) {
      row_weights(x, s, pah, pal);
      return;
    }
  }
  auto scores = [&](float ref) {
    row_scores(a, scale2, slope, sloped, mylen - 1 - key0, ref, x);
    if (!plain) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = key0 + i;
        const bool in = (key < mylen) & (key >= mylo) & ((key >= mywlo) | (key < keep));
        x[i] = in ? x[i] : -INFINITY;
      }
    }
  };
  scores(s.ref);
  float mx = top8(x);
  if (__any(mx > s.rise)) {
    mx = row_max(mx);
    const bool up = mx > s.rise;
    const float ref = up ? s.ref + mx : s.ref;
    const float corr = s.rise < 0.f ? 1.f : __builtin_amdgcn_exp2f(s.ref - ref);  // (nothing summed yet: nothing to correct)
#pragma unroll
    for (int n = 0; n < NCB; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[n][r] *= corr;
    s.l *= corr;
    s.ref = ref;
    if (up) s.rise = RISE;
    scores(ref);
  }
  row_weights(x, s, pah, pal);
}
// the tile's key that row r of the score product's block kb is: lanes come to hold neighbours
__device__ __forceinline__ int dealt_key(int r, int kb) { return 8 * (r >> 2) + 4 * kb + (r & 3); }

}  // namespace sm
