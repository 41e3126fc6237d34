// Latent attention of any size over a paged latent cache (one row [latent R | rotated key dr]
// per token, shared by all heads).
//
// latent_rope_cache: rotate the query's rotary part (pairs (i, i + rot_dims/2) or (2i, 2i+1) over
//   the first rot_dims dimensions, angles from an fp32 cos/sin table) into the absorbed query, RMS-norm
//   the latent with its plain weight, rotate the shared key part and write the cache row. A layer
//   that reads another layer's cache passes no kv and rotates its queries only.
// All attention forms take an optional gate [T, H]: head h's result times sigmoid(gate[t, h]).
// latent_attention: one workgroup = QT consecutive token rows x 4 heads (one wave per head).
//   Keys stream through LDS in tiles of KT rows (fp32) shared by all 4 x QT (row, head) pairs;
//   a lane scores one key (dot over R + dr from LDS), the wave keeps an online softmax per pair,
//   and the lanes then own output columns for the P x latent product. Scores, softmax and the
//   accumulators are fp32. A row's result depends only on its own keys and the fixed tile
//   size, never on what else is in the step.
// window > 0: query i sees key j <= i only if i - j < window; the tiles before the first window of a
//   work item are not visited (tiles start at multiples of the tile size from position 0). dr may be 0: a
//   latent without a rotated part.
#include "row_softmax.h"
#include "seqmix_common.h"

using namespace sm;

namespace {

constexpr int NT = 256;

template <typename T>
__global__ __launch_bounds__(NT) void latent_rope_cache_kernel(
    const T* __restrict__ q, int64_t q_stride, const T* __restrict__ kv, int64_t kv_stride,
    const T* __restrict__ norm_w, float eps, const int64_t* __restrict__ positions,
    const float* __restrict__ cos_sin, int H, int dn, int dr, int rot_dims, int R,
    const int64_t* __restrict__ slots, T* __restrict__ cache, T* __restrict__ q_abs, int interleaved) {
  __shared__ float red[NT / 64];
  const int64_t t = blockIdx.x;
  const int half = rot_dims >> 1;
  const float* cs = cos_sin + positions[t] * rot_dims;  // [cos(half) | sin(half)]
  const int Dk = R + dr;
  // element i of a rotated vector at src
  auto rot = [&](const T* src, int i) {
    if (i >= rot_dims) return ld(src + i);
    if (interleaved) {
      const int f = i >> 1;
      return (i & 1) ? ld(src + i) * cs[f] + ld(src + i - 1) * cs[half + f]
                     : ld(src + i) * cs[f] - ld(src + i + 1) * cs[half + f];
    }
    return i < half ? ld(src + i) * cs[i] - ld(src + i + half) * cs[half + i]
                    : ld(src + i) * cs[i - half] + ld(src + i - half) * cs[i];
  };
  // query: rotary part of every head -> q_abs[t, h, R + i]
  for (int e = threadIdx.x; e < H * dr; e += NT) {
    const int h = e / dr, i = e - h * dr;
    st(q_abs + (t * H + h) * Dk + R + i, rot(q + t * q_stride + (int64_t)h * (dn + dr) + dn, i));
  }
  if (kv == nullptr) return;
  // latent: RMS norm with a plain weight
  const T* kr = kv + t * kv_stride;
  float ss = 0.f;
  for (int c = threadIdx.x; c < R; c += NT) {
    const float v = ld(kr + c);
    ss += v * v;
  }
  ss = block_sum<NT>(ss, red);
  const int64_t slot = slots[t];
  if (slot < 0) return;
  const float inv = 1.f / sqrtf(ss / (float)R + eps);
  T* row = cache + slot * Dk;
  for (int c = threadIdx.x; c < R; c += NT) st(row + c, ld(kr + c) * inv * ld(norm_w + c));
  for (int i = threadIdx.x; i < dr; i += NT) st(row + R + i, rot(kr + R, i));
}

// RC = ceil(R / 64) output columns per lane; QT token rows per workgroup.
template <typename T, int RC, int QT>
__global__ __launch_bounds__(NT) void latent_attention_kernel(
    const T* __restrict__ q_abs, const T* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
    const int* __restrict__ row_seq, const int* __restrict__ row_len, float scale, int H, int R, int Dk, int KT,
    int T_rows, T* __restrict__ out, const T* __restrict__ gate, int64_t gate_stride, int window) {
  extern __shared__ float lds[];
  const int KS = Dk + 1;                 // key row stride in LDS (odd: lanes hit distinct banks)
  float* sK = lds;                       // [KT][KS]
  float* sQ = lds + KT * KS;             // [QT][4][Dk], pre-scaled
  const int t0 = blockIdx.x * QT;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int h = blockIdx.y * 4 + wave;
  const bool head_ok = h < H;

  for (int e = threadIdx.x; e < QT * 4 * Dk; e += NT) {
    const int r = e / (4 * Dk), rem = e - r * 4 * Dk;
    const int w = rem / Dk, d = rem - w * Dk;
    const int t = t0 + r, hh = blockIdx.y * 4 + w;
    sQ[e] = (t < T_rows && hh < H) ? ld(q_abs + ((int64_t)t * H + hh) * Dk + d) * scale : 0.f;
  }

  int seq_r[QT], len_r[QT], lo_r[QT];
  bool done[QT];
#pragma unroll
  for (int r = 0; r < QT; ++r) {
    const int t = t0 + r;
    done[r] = t >= T_rows;
    seq_r[r] = done[r] ? -1 : row_seq[t];
    len_r[r] = done[r] ? 0 : row_len[t];
    lo_r[r] = window > 0 ? max(0, len_r[r] - window) : 0;  // first key of the row's window
  }

  for (int pass = 0; pass < QT; ++pass) {
    // rows of this pass: those of the first unfinished row's sequence
    int seq = -1;
#pragma unroll
    for (int r = 0; r < QT; ++r)
      if (seq < 0 && !done[r]) seq = seq_r[r];
    if (seq < 0) break;
    bool act[QT];
    int maxlen = 0, minlo = 0x7fffffff;
#pragma unroll
    for (int r = 0; r < QT; ++r) {
      act[r] = !done[r] && seq_r[r] == seq;
      if (act[r]) {
        maxlen = max(maxlen, len_r[r]);
        minlo = min(minlo, lo_r[r]);
      }
    }
    float m[QT], l[QT], acc[QT][RC];
#pragma unroll
    for (int r = 0; r < QT; ++r) {
      m[r] = -INFINITY;
      l[r] = 0.f;
#pragma unroll
      for (int c = 0; c < RC; ++c) acc[r][c] = 0.f;
    }
    const int* bt = tables + (int64_t)seq * W;
    for (int k0 = (minlo / KT) * KT; k0 < maxlen; k0 += KT) {
      __syncthreads();  // previous tile fully used (and sQ written, first time)
      for (int e = threadIdx.x; e < KT * Dk; e += NT) {
        const int j = e / Dk, d = e - j * Dk;
        const int key = k0 + j;
        float v = 0.f;
        if (key < maxlen) {
          const int64_t rowi = (int64_t)bt[key / bs] * bs + (key % bs);
          v = ld(cache + rowi * Dk + d);
        }
        sK[j * KS + d] = v;
      }
      __syncthreads();
      if (!head_ok) continue;
#pragma unroll
      for (int r = 0; r < QT; ++r) {
        if (!act[r] || k0 >= len_r[r] || k0 + KT <= lo_r[r]) continue;
        const bool valid = lane < KT && k0 + lane < len_r[r] && k0 + lane >= lo_r[r];
        float s = -INFINITY;
        if (valid) {
          const float* qv = sQ + (r * 4 + wave) * Dk;
          const float* kr = sK + lane * KS;
          float a = 0.f;
          for (int d = 0; d < Dk; ++d) a += qv[d] * kr[d];
          s = a;
        }
        const float mn = fmaxf(m[r], wave_max(s));
        const float corr = expf(m[r] - mn);  // exp(-inf) = 0 on the first tile
        const float p = valid ? expf(s - mn) : 0.f;
        l[r] = l[r] * corr + wave_sum(p);
        m[r] = mn;
#pragma unroll
        for (int c = 0; c < RC; ++c) acc[r][c] *= corr;
        const int nk = min(KT, len_r[r] - k0);
        for (int j = max(0, lo_r[r] - k0); j < nk; ++j) {
          const float pj = __shfl(p, j, 64);
          const float* kr = sK + j * KS;
#pragma unroll
          for (int c = 0; c < RC; ++c) {
            const int col = lane + 64 * c;
            if (col < R) acc[r][c] += pj * kr[col];
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < QT; ++r) {
      if (!act[r]) continue;
      done[r] = true;
      if (!head_ok) continue;
      float inv = 1.f / l[r];
      if (gate) inv *= 1.f / (1.f + expf(-ld(gate + (int64_t)(t0 + r) * gate_stride + h)));
#pragma unroll
      for (int c = 0; c < RC; ++c) {
        const int col = lane + 64 * c;
        if (col < R) st(out + ((int64_t)(t0 + r) * H + h) * R + col, acc[r][c] * inv);
      }
    }
  }
}


// ---------------------------------------------------------------------------------------------
// bf16 forms on the matrix cores. A workgroup takes one work item: up to 64 (token, head) rows of
// ONE sequence (consecutive tokens x all heads). Keys stream through LDS row-major; the scores are
// S^T = K Q^T (v_mfma_f32_16x16x32_bf16, fp32 accumulation of exact bf16 products) and the latent part
// of the same tile is the second product's B operand, read transposed (ds_read_b64_tr_b16: 16 lanes
// read 4 keys x 16 columns, a lane gets one column's four keys). Softmax is fp32 per row in base 2;
// the weights P enter the second product as a bf16 pair (hi + lo, two MFMAs), which keeps 16 mantissa
// bits of the fp32 weight. DkP = 32 NKS >= Dk >= R are the padded sizes (zeros in LDS and in the
// query fragments); columns past R are computed from whatever the row holds there and not stored.
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));

constexpr float LOG2E = 1.44269504088896341f;

// Eight keys of one column for a lane: four from ``p`` on and four from ROWS rows further down.
template <int KS, int ROWS = 16>
__device__ __forceinline__ bf16x8_t column_keys(const bf16_t* p) {
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + ROWS * KS));
  return __builtin_bit_cast(bf16x8_t, s16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}

// Softmax weights of eight keys (fp32) as the bf16 pair hi + lo: hi = the upper 16 bits (truncated), lo = the
// upper 16 bits of the exact rest, so hi + lo differs from the weight by less than 2^-16 of it.
__device__ __forceinline__ void split_weights(const float* p, bf16x8_t& hi, bf16x8_t& lo) {
  u32x4_t hw, lw;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float p0 = p[2 * i], p1 = p[2 * i + 1];
    const uint32_t u0 = __float_as_uint(p0), u1 = __float_as_uint(p1);
    const uint32_t r0 = __float_as_uint(p0 - __uint_as_float(u0 & 0xffff0000u));
    const uint32_t r1 = __float_as_uint(p1 - __uint_as_float(u1 & 0xffff0000u));
    hw[i] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // the upper halves of both
    lw[i] = __builtin_amdgcn_perm(r1, r0, 0x07060302u);
  }
  hi = __builtin_bit_cast(bf16x8_t, hw);
  lo = __builtin_bit_cast(bf16x8_t, lw);
}

// Keys of a range: one tile while that makes up to 32 ranges (the merge is longer with more), else two. A tile takes a decode
// workgroup 4.5 us, most of it waiting for its keys: 9 rows of 577 to 1777 keys, 16 heads, with the merge 27.4 us in ranges of 192,
// 23.3 of 64; one of 300 25.5 / 17.0; 16 of up to 300 25.2 / 16.6; four of 8000 keep theirs of 128, 27.1 (30.8 of 64).
__device__ __forceinline__ int least_keys(const int* longest) { return longest != nullptr && *longest <= 32 * 64 ? 64 : 128; }

// One tile's rows of the paged cache, in 16-byte chunks with the lanes along a row: KEYS keys from k0 on, zeros from
// kend on and past Dk. All chunks are requested before any is used. one_page: the tile lies inside one
// page (page sizes that are multiples of KEYS), so its block-table entry is read once.
template <int KEYS, int DkP>
struct TileFetch {
  static constexpr int CPR = DkP / 8, NCH = (KEYS * CPR + NT - 1) / NT, KS = DkP + 8;
  u32x4_t v[NCH];
  // The thread's number, opaque to the optimiser: the chunks' places are recomputed for every tile (two or
  // three instructions each) instead of being kept in registers across the loop.
  static __device__ __forceinline__ int here() {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
  }
  __device__ __forceinline__ void load(const bf16_t* cache, const int* bt, int bs, int Dk, int k0, int kend) {
    const int tid = here();
    const bool one_page = (bs % KEYS) == 0, vec = (Dk & 7) == 0;
    const int64_t row0 = one_page ? (int64_t)bt[k0 / bs] * bs + (k0 % bs) : 0;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int e = tid + i * NT;
      const int j = e / CPR, c = e - j * CPR;
      const int key = k0 + j;
      u32x4_t t = {0, 0, 0, 0};
      if (e < KEYS * CPR && key < kend && c * 8 < Dk) {
        const int64_t row = one_page ? row0 + j : (int64_t)bt[key / bs] * bs + (key % bs);
        const bf16_t* src = cache + row * Dk + c * 8;
        if (vec) {
          t = *reinterpret_cast<const u32x4_t*>(src);
        } else {
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (c * 8 + q < Dk) t[q >> 1] |= (uint32_t)src[q] << (16 * (q & 1));
        }
      }
      v[i] = t;
    }
  }
  __device__ __forceinline__ void store(bf16_t* tile) const {
    const int tid = here();
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int e = tid + i * NT;
      const int j = e / CPR, c = e - j * CPR;
      if (e < KEYS * CPR) *reinterpret_cast<u32x4_t*>(&tile[j * KS + c * 8]) = v[i];
    }
  }
};

// The wide form (Dk = 32 NKS = 512 or 576 exactly, R <= 512, pages of whole tiles): the accumulators and the query leave no
// buffer holds 128 bytes of all 32 rows, then the next 128; eight pieces of 16 bytes lie in the order c ^ f(row). f is even, so that
// the pairs of pieces that a transposed read takes stay together, and neither of the two kinds of reads meets in a bank: lanes 0 .. 3
// and 12 .. 15 of a 16-byte read go with lanes 4 .. 11 of the quarter beside theirs, a transposed one takes eight neighbouring rows.
// The second product comes out as O^T, in the lanes that own the rows (see grouped_attention_mfma). 2048 tokens, 16 heads, latent
// 512 + 64: 299 us with the general form below (a tile's loads were waited for in the loop; items in order of their length), 149 with
// the query waited for in the loop, and the next tile with it, and conflicts in a third of the transposed reads' cycles, now 142.
template <int NKS>
__global__ __launch_bounds__(NT, 2) void latent_prompt_kernel(
    const bf16_t* __restrict__ q_abs, const bf16_t* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
    const int* __restrict__ items, const int* __restrict__ row_len, float scale, int H, int R, bf16_t* __restrict__ out,
    const bf16_t* __restrict__ gate, int64_t gate_stride, int window) {
  constexpr int Dk = 32 * NKS, NCB = 32, RB = 2 * Dk, NG = RB / 128;  // bytes of a row, its parts of 128
  static_assert(NKS % 2 == 0, "whole parts");
  __shared__ __attribute__((aligned(1024))) char tile[2 * MKT * RB];
  auto f = [](int row) { return row & 6; };
  const int seq = items[blockIdx.x * 3], tok0 = items[blockIdx.x * 3 + 1], ntok = items[blockIdx.x * 3 + 2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  // this lane's query row: item row 16 wave + r16
  const int myrow = wave * 16 + r16;
  const bool row_ok = myrow < ntok * H;
  const int mytok = tok0 + (row_ok ? myrow / H : 0), myhead = row_ok ? myrow % H : 0;
  const int mylen = row_ok ? row_len[mytok] : 0;
  const int mylo = window > 0 ? max(0, mylen - window) : 0;  // first key of the row's window
  const int kend = row_len[tok0 + ntok - 1];                 // the run's last token sees the most keys
  // the run's first token has the earliest window; tiles start at multiples of 32 from position 0
  const int kbeg = window > 0 ? (max(0, row_len[tok0] - window) / MKT) * MKT : 0;
  // tiles in [full_lo, full_hi) are visible to every row of the item: no mask
  const int full_lo = window > 0 ? max(0, kend - window) : 0, full_hi = row_len[tok0];

  bf16x8_t qf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    qf[ks] = *reinterpret_cast<const bf16x8_t*>(q_abs + ((int64_t)mytok * H + myhead) * Dk + ks * 32 + kq * 8);
  f32x4_t o[NCB];  // o[n][r] = this lane's row, column 16 n + 4 kq + r
#pragma unroll
  for (int n = 0; n < NCB; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // the weights' reference (base 2), the sum over this lane's keys
  const int* bt = tables + (int64_t)seq * W;
  const float scale2 = scale * LOG2E;
  const bool pow2 = (bs & (bs - 1)) == 0;
  const int sh = __builtin_ctz(bs);
  auto page_of = [&](int k0) { return k0 < kend ? bt[pow2 ? k0 >> sh : k0 / bs] : 0; };

  // places inside a buffer: this lane's pieces of the first product's rows, and of the transposed reads
  int ka[2], va[4];
#pragma unroll
  for (int e = 0; e < 2; ++e) ka[e] = r16 * 128 + ((e * 4 + kq) ^ f(r16)) * 16;
  const int vrow = 4 * kq + (r16 >> 2);
#pragma unroll
  for (int j = 0; j < 4; ++j) va[j] = vrow * 128 + ((r16 >> 1 & 1) ^ f(vrow) ^ 2 * j) * 16 + (r16 & 1) * 8;
  // a wave copies eight rows, eight lanes per row and part
  const int crow = wave * 8 + (lane >> 3), cpiece = ((lane & 7) ^ f(crow)) * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tile + wave * 1024;
  int page = page_of(kbeg);
  auto copy = [&](int k0, int buf) {
    const char* base = reinterpret_cast<const char*>(cache + ((int64_t)page * bs + (pow2 ? k0 & (bs - 1) : k0 % bs)) * Dk);
    page = page_of(k0 + MKT);
    // keys past the end: the last one again (a page's unwritten rest may hold anything)
    const uint32_t off = min(crow, kend - 1 - k0) * RB + cpiece;
#pragma unroll
    for (int i = 0; i < NG; ++i) copy_1k(base + i * 128, off, lds0 + buf * (MKT * RB) + i * (MKT * 128));
  };
  auto arrive = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  if (kbeg < kend) copy(kbeg, 0);
  // (a wait that hipcc sees, though not the copies: where the query might be pending at the loop's entry it would wait for all in the loop)
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");  // (neither is a fence for hipcc: reads of the tile stay below)
  int cur = 0;
  for (int k0 = kbeg; k0 < kend; k0 += MKT, cur ^= 1) {
    const char* const t = tile + cur * (MKT * RB);
    if (k0 + MKT < kend) copy(k0 + MKT, cur ^ 1);  // read by nobody since the barrier of the previous tile
    // scores of this lane's row against keys k0 + 16 kb + 4 kq + r
    float sc[8];
    {
      f32x4_t a[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const bf16x8_t k = *reinterpret_cast<const bf16x8_t*>(t + ka[ks & 1] + (ks >> 1) * (MKT * 128) + kb * 16 * 128);
          a[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[ks], a[kb], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < 8; ++i) sc[i] = a[i >> 2][i & 3] * scale2;
    }
    if (k0 < full_lo || k0 + MKT > full_hi) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = k0 + (i >> 2) * 16 + kq * 4 + (i & 3);
        sc[i] = ((key < mylen) & (key >= mylo)) ? sc[i] : -INFINITY;
      }
    }
    float mx = sc[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, sc[i]);
    mx = row_max(mx);
    // the reference moves only when a score of the row passes it by 2^8: weights of up to 2^8 lose nothing in fp32. The branch
    // is the wave's, the move the row's own: other rows of the wave are multiplied by 1
    if (__any(mx > m + 8.f)) {
      const float mn = mx > m + 8.f ? mx : m;
      const float corr = mn == m ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      l *= corr;
      m = mn;
#pragma unroll
      for (int n = 0; n < NCB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] *= corr;
    }
    const float mref = m == -INFINITY ? 0.f : m;  // a row with no key yet
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[i] = __builtin_amdgcn_exp2f(sc[i] - mref);
      l += sc[i];
    }
    bf16x8_t pah, pal;
    split_weights(sc, pah, pal);
#pragma unroll
    for (int n0 = 0; n0 < NCB; n0 += 4) {
      bf16x8_t v[4];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        v[n] = column_keys<64>(reinterpret_cast<const bf16_t*>(t + va[n] + (n0 >> 2) * (MKT * 128)));
#pragma unroll
      for (int n = 0; n < 4; ++n) o[n0 + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[n], pah, o[n0 + n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 4; ++n) o[n0 + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[n], pal, o[n0 + n], 0, 0, 0);
    }
    arrive();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!row_ok) return;
  float w = 1.f / l;
  if (gate) w *= 1.f / (1.f + expf(-ld(gate + (int64_t)mytok * gate_stride + myhead)));
  bf16_t* dst = out + ((int64_t)mytok * H + myhead) * R;
#pragma unroll
  for (int n = 0; n < NCB; ++n) {
    const int col = n * 16 + kq * 4;
    if (col + 4 <= R && (R & 3) == 0) {
      ushort4 b;
      st(&b.x, o[n][0] * w); st(&b.y, o[n][1] * w); st(&b.z, o[n][2] * w); st(&b.w, o[n][3] * w);
      *reinterpret_cast<ushort4*>(dst + col) = b;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (col + r < R) st(dst + col + r, o[n][r] * w);
    }
  }
}

// Prompts with keys and values of their own. A prompt's rows meet so many keys that the heads' keys W_uk c and values W_uv c are
// cheaper made once than absorbed into every query: 192 + 128 columns per head and key instead of 576 + 512. The latents of the
// prompts' sequences are gathered out of their pages, one product makes [key | value] of every head, and the rotated part stays shared.
// The tiles lie in LDS as in latent_prompt_kernel, in parts of 128 bytes of all 32 keys: two of the head's key, the rotated part, two of
// the values; key rows are dealt as in grouped_prompt_kernel (f(row): no bank conflicts for either kind of read in that order), whose
// softmax this is. What bounds it: the waves' latency (QK, softmax, PV in a row, three to four waves per SIMD).
// 2048 tokens, 16 heads, latent 512 + 64, values 128, us: the absorbed form's kernel and the products before and behind it 19 + 142 + 16,
// here gather, product, kernel 4 + 20 + 64; 0.0023 off 64 bits (0.0024).
constexpr int OWN_K = 128, OWN_ROT = 64, OWN_V = 128;
__global__ __launch_bounds__(NT, 4) void latent_own_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ q_rot, int64_t rot_stride, int64_t rot_head,
    const bf16_t* __restrict__ kv, const bf16_t* __restrict__ rot, const int* __restrict__ base, const int* __restrict__ items,
    const int* __restrict__ row_len, float scale, int H, bf16_t* __restrict__ out, int64_t out_stride, const bf16_t* __restrict__ gate,
    int64_t gate_stride) {
  constexpr int NKS = (OWN_K + OWN_ROT) / 32, NCB = OWN_V / 16, PART = MKT * 128, TB = 5 * PART;
  __shared__ __attribute__((aligned(1024))) char tile[2 * TB];
  auto f = [](int row) { return (row & 2) | (row >> 1 & 4); };
  const int h = blockIdx.x;
  const int seq = items[blockIdx.y * 3], tok0 = items[blockIdx.y * 3 + 1], ntok = items[blockIdx.y * 3 + 2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  const int myrow = wave * 16 + r16;
  const bool ok = myrow < ntok;
  const int mytok = tok0 + (ok ? myrow : 0);
  const int mylen = ok ? row_len[mytok] : 0;
  const int kend = row_len[tok0 + ntok - 1], full = row_len[tok0];  // tiles below ``full`` are visible to every row

  bf16x8_t qf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    qf[ks] = *reinterpret_cast<const bf16x8_t*>(ks < OWN_K / 32 ? q + mytok * q_stride + h * (OWN_K + OWN_ROT) + ks * 32 + kq * 8
                                                                : q_rot + mytok * rot_stride + h * rot_head + (ks - OWN_K / 32) * 32 + kq * 8);
  RowSoftmax sm;
  sm.start(nullptr, 0, kq);
  f32x4_t o[NCB];
#pragma unroll
  for (int n = 0; n < NCB; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float scale2 = scale * LOG2E;

  // a wave copies eight rows of every part, eight lanes per row
  const int crow = wave * 8 + (lane >> 3), cpiece = ((lane & 7) ^ f(crow)) * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tile + wave * 1024;
  const int64_t pitch = (int64_t)H * (OWN_K + OWN_V) * 2;  // bytes of a row of kv
  const char* const kv0 = reinterpret_cast<const char*>(kv) + base[seq] * pitch + h * (OWN_K + OWN_V) * 2;
  const char* const rot0 = reinterpret_cast<const char*>(rot) + (int64_t)base[seq] * (OWN_ROT * 2);
  auto copy = [&](int k0, int buf) {
    const int row = min(crow, kend - 1 - k0);  // rows past the end: the last one again
    const uint32_t off = (uint32_t)(row * pitch) + cpiece, at = lds0 + buf * TB;
    const char* const b = kv0 + k0 * pitch;
    copy_1k(b, off, at);
    copy_1k(b + 128, off, at + PART);
    copy_1k(rot0 + k0 * (OWN_ROT * 2), row * (OWN_ROT * 2) + cpiece, at + 2 * PART);
    copy_1k(b + OWN_K * 2, off, at + 3 * PART);
    copy_1k(b + OWN_K * 2 + 128, off, at + 4 * PART);
  };
  int ka[2], va[4];
  const int krow = dealt_key(r16, 0), vrow = 8 * kq + (r16 >> 2);
#pragma unroll
  for (int e = 0; e < 2; ++e) ka[e] = krow * 128 + ((e * 4 + kq) ^ f(krow)) * 16;
#pragma unroll
  for (int j = 0; j < 4; ++j) va[j] = 3 * PART + vrow * 128 + ((r16 >> 1 & 1) ^ f(vrow) ^ 2 * j) * 16 + (r16 & 1) * 8;
  copy(0, 0);
  // (a wait that hipcc sees, though not the copies: where the query might be pending at the loop's entry it would wait for all in the loop)
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");  // (neither is a fence for hipcc: reads of the tile stay below)
  int cur = 0;
  for (int k0 = 0; k0 < kend; k0 += MKT, cur ^= 1) {
    const char* const t = tile + cur * TB;
    if (k0 + MKT < kend) copy(k0 + MKT, cur ^ 1);  // read by nobody since the barrier of the previous tile
    f32x4_t a[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const bf16x8_t k = *reinterpret_cast<const bf16x8_t*>(t + ka[ks & 1] + (ks >> 1) * PART + kb * 4 * 128);
        a[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[ks], a[kb], 0, 0, 0);
      }
    bf16x8_t pah, pal;
    weigh<NCB, true>(a, scale2, 0.f, false, k0 + MKT <= full, k0 + kq * 8, mylen, 0, 0, 0, sm, o, pah, pal);
#pragma unroll
    for (int n0 = 0; n0 < NCB; n0 += 4) {
      bf16x8_t v[4];
#pragma unroll
      for (int n = 0; n < 4; ++n)
        v[n] = column_keys<64, 4>(reinterpret_cast<const bf16_t*>(t + va[n] + (n0 >> 2) * PART));
#pragma unroll
      for (int n = 0; n < 4; ++n) o[n0 + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[n], pah, o[n0 + n], 0, 0, 0);
#pragma unroll
      for (int n = 0; n < 4; ++n) o[n0 + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[n], pal, o[n0 + n], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  const float l = row_sum(sm.l);
  if (!ok) return;
  float w = 1.f / l;
  if (gate) w *= 1.f / (1.f + expf(-ld(gate + (int64_t)mytok * gate_stride + h)));
  bf16_t* dst = out + mytok * out_stride + h * OWN_V;
#pragma unroll
  for (int n = 0; n < NCB; ++n) {
    ushort4 b;
    st(&b.x, o[n][0] * w); st(&b.y, o[n][1] * w); st(&b.z, o[n][2] * w); st(&b.w, o[n][3] * w);
    *reinterpret_cast<ushort4*>(dst + n * 16 + kq * 4) = b;
  }
}

// Cached rows [R | dr] of the sequences ``seq`` .. (blockIdx.y further), back to back from base[seq] on: the latents and the rotated
// parts apart. base has one number more than there are sequences.
__global__ __launch_bounds__(NT) void latent_gather_kernel(const bf16_t* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
                                                           const int* __restrict__ base, int first, int R, int dr,
                                                           bf16_t* __restrict__ lat, bf16_t* __restrict__ rot) {
  const int seq = first + blockIdx.y, b = base[seq], n = base[seq + 1] - b, pieces = (R + dr) >> 3;
  const int e = blockIdx.x * NT + threadIdx.x, key = e / pieces, c = (e - key * pieces) * 8;
  if (key >= n) return;
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(cache + ((int64_t)tables[(int64_t)seq * W + key / bs] * bs + key % bs) * (R + dr) + c);
  bf16_t* dst = c < R ? lat + (int64_t)(b + key) * R + c : rot + (int64_t)(b + key) * dr + c - R;
  *reinterpret_cast<u32x4_t*>(dst) = v;
}

// 16 rows per wave, every wave over all columns. Two tile buffers: the next tile is written while the
// current one is read, one barrier per tile. The weights never leave the registers: after S^T = K Q^T a
// lane holds, for its query row, the keys 4 kq .. 4 kq + 3 of both 16-key halves, which is one A operand
// of the second product with the contraction in that order - the order the transposed reads deliver.
template <int NKS, int NCB>
__global__ __launch_bounds__(NT, 2) void latent_attention_mfma_kernel(
    const bf16_t* __restrict__ q_abs, const bf16_t* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
    const int* __restrict__ items, const int* __restrict__ row_len, float scale, int H, int R, int Dk,
    bf16_t* __restrict__ out, int split_keys, float* __restrict__ part_o, float* __restrict__ part_ml,
    const bf16_t* __restrict__ gate, int64_t gate_stride, int window, const int* __restrict__ longest) {
  constexpr int DkP = 32 * NKS;
  static_assert(16 * NCB <= DkP, "columns inside the row");
  // the largest forms have no registers left to keep a tile in flight: their two workgroups per CU overlap
  constexpr bool PRE = NKS <= 10;
  using Tile = TileFetch<MKT, DkP>;
  constexpr int KS = Tile::KS;  // LDS row stride (bf16), a multiple of 16 bytes
  __shared__ __attribute__((aligned(16))) bf16_t sK[2 * MKT * KS];
  const int seq = items[blockIdx.x * 3], tok0 = items[blockIdx.x * 3 + 1], ntok = items[blockIdx.x * 3 + 2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  // this lane's query row (as the B operand's column): item row 16 wave + r16
  const int myrow = wave * 16 + r16;
  const bool row_ok = myrow < ntok * H;
  const int mytok = tok0 + (row_ok ? myrow / H : 0), myhead = row_ok ? myrow % H : 0;
  const int mylen = row_ok ? row_len[mytok] : 0;
  const int mylo = window > 0 ? max(0, mylen - window) : 0;  // first key of the row's window
  const int maxlen = row_len[tok0 + ntok - 1];  // the run's last token sees the most keys
  // the run's first token has the earliest window; tiles start at multiples of 32 from position 0
  const int kbase = window > 0 ? (max(0, row_len[tok0] - window) / MKT) * MKT : 0;

  bf16x8_t qf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int d = ks * 32 + kq * 8 + i;
      const bf16_t w = (row_ok && d < Dk) ? q_abs[((int64_t)mytok * H + myhead) * Dk + d] : (bf16_t)0;
      qf[ks][i] = __builtin_bit_cast(__bf16, w);
    }
  }
  f32x4_t o[NCB];
#pragma unroll
  for (int n = 0; n < NCB; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int* bt = tables + (int64_t)seq * W;
  const float scale2 = scale * LOG2E;
  // decode steps split a row's keys over blockIdx.y: this workgroup takes [kbeg, kend)
  const int nsplit = gridDim.y;
  if (nsplit > 1) {
    if ((int)blockIdx.y >= ranges_used(longest, nsplit, split_keys, least_keys(longest))) return;
    split_keys = range_keys(longest, nsplit, split_keys, least_keys(longest));
  }
  const int kbeg = nsplit > 1 ? kbase + blockIdx.y * split_keys : kbase;
  const int kend = nsplit > 1 ? min(maxlen, kbeg + split_keys) : maxlen;
  const int voff = (4 * kq + (r16 >> 2)) * KS + 4 * (r16 & 3);  // this lane's part of a transposed read
  // tiles in [full_lo, full_hi) are visible to every row of the item: no mask
  const int full_lo = window > 0 ? max(0, maxlen - window) : 0, full_hi = min(row_len[tok0], kend);

  Tile tf;
  if (kbeg < kend) {
    tf.load(cache, bt, bs, Dk, kbeg, kend);
    tf.store(sK);
  }
  __syncthreads();
  int cur = 0;
  for (int k0 = kbeg; k0 < kend; k0 += MKT, cur ^= 1) {
    const bf16_t* const tK = sK + cur * MKT * KS;
    const bool more = k0 + MKT < kend;
    if (PRE && more) tf.load(cache, bt, bs, Dk, k0 + MKT, kend);  // in flight during this tile's products
    // scores of this lane's row against keys k0 + 16 kb + 4 kq + r
    float sc[8];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x4_t a = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const bf16x8_t ka = *reinterpret_cast<const bf16x8_t*>(&tK[(kb * 16 + r16) * KS + ks * 32 + kq * 8]);
        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[ks], a, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[kb * 4 + r] = a[r] * scale2;
    }
    if (k0 < full_lo || k0 + MKT > full_hi) {
      const int hi = min(mylen, kend);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = k0 + (i >> 2) * 16 + kq * 4 + (i & 3);
        sc[i] = ((key < hi) & (key >= mylo)) ? sc[i] : -INFINITY;
      }
    }
    float mx = sc[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, sc[i]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const float mref = (mn == -INFINITY) ? 0.f : mn;  // a row with no key yet
    const float corr = __builtin_amdgcn_exp2f(m - mref);
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[i] = __builtin_amdgcn_exp2f(sc[i] - mref);
      psum += sc[i];
    }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l = l * corr + psum;
    m = mn;
    bf16x8_t pah, pal;
    split_weights(sc, pah, pal);
    if (__any(corr != 1.f)) {  // wave-uniform: some row's maximum moved in this tile
      // the accumulators hold rows 4 kq + r: their correction comes from the lane that owns the row
      float cr[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) cr[r] = __shfl(corr, kq * 4 + r, 64);
#pragma unroll
      for (int n = 0; n < NCB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] *= cr[r];
    }
#pragma unroll
    for (int n = 0; n < NCB; ++n) {
      const bf16x8_t vb = column_keys<KS>(tK + voff + n * 16);
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pah, vb, o[n], 0, 0, 0);
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pal, vb, o[n], 0, 0, 0);
    }
    // every wave has finished the previous tile (barrier below, one iteration ago), so the other buffer is free
    if (!PRE && more) tf.load(cache, bt, bs, Dk, k0 + MKT, kend);
    if (more) tf.store(sK + (cur ^ 1) * MKT * KS);
    __syncthreads();
  }
  // o[n][r] = O[row 4 kq + r][column 16 n + r16]
  if (nsplit > 1) {
    // partial result of this key range: unnormalised o, with the row's running max (base 2) and sum
    const int64_t pbase = ((int64_t)blockIdx.x * nsplit + blockIdx.y) * 64;
    if (kq == 0) {
      part_ml[(pbase + myrow) * 2] = m;
      part_ml[(pbase + myrow) * 2 + 1] = l;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wave * 16 + kq * 4 + r;
#pragma unroll
      for (int n = 0; n < NCB; ++n) {
        const int col = n * 16 + r16;
        if (col < R) part_o[(pbase + row) * R + col] = o[n][r];
      }
    }
    return;
  }
  float inv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = 1.f / __shfl(l, kq * 4 + r, 64);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = wave * 16 + kq * 4 + r;
    if (row >= ntok * H) continue;
    const int64_t base = ((int64_t)(tok0 + row / H) * H + row % H) * R;
    float w = inv[r];
    if (gate) w *= 1.f / (1.f + expf(-ld(gate + (int64_t)(tok0 + row / H) * gate_stride + row % H)));
#pragma unroll
    for (int n = 0; n < NCB; ++n) {
      const int col = n * 16 + r16;
      if (col < R) st(out + base + col, o[n][r] * w);
    }
  }
}

// Steps of single tokens: an item has few rows, so the four waves share them. A workgroup takes 16 rows
// (blockIdx.z: which of the item's) and tiles of 64 keys: wave w scores keys 16 w .. 16 w + 15, the
// scores meet in LDS, every wave forms the 16 x 64 softmax weights from there and multiplies them with
// its quarter of the columns. The next tile's loads are in flight from one tile's staging to the next.
constexpr int DKT = 64;
template <int NKS, int NCW>
__global__ __launch_bounds__(NT, 2) void latent_decode_mfma_kernel(
    const bf16_t* __restrict__ q_abs, const bf16_t* __restrict__ cache, const int* __restrict__ tables, int W, int bs,
    const int* __restrict__ items, const int* __restrict__ row_len, float scale, int H, int R, int Dk,
    bf16_t* __restrict__ out, int split_keys, float* __restrict__ part_o, float* __restrict__ part_ml,
    const bf16_t* __restrict__ gate, int64_t gate_stride, int window, const int* __restrict__ longest) {
  constexpr int DkP = 32 * NKS;
  static_assert(64 * NCW <= DkP, "columns inside the row");
  using Tile = TileFetch<DKT, DkP>;
  constexpr int KS = Tile::KS, SS = DKT + 4;
  __shared__ __attribute__((aligned(16))) bf16_t sK[DKT * KS];
  __shared__ __attribute__((aligned(16))) float sS[16 * SS];  // scores [row][key], base 2, masked
  const int seq = items[blockIdx.x * 3], tok0 = items[blockIdx.x * 3 + 1], ntok = items[blockIdx.x * 3 + 2];
  const int row0 = blockIdx.z * 16;
  if (row0 >= ntok * H) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  const int myrow = row0 + r16;  // this lane's query row
  const bool row_ok = myrow < ntok * H;
  const int mytok = tok0 + (row_ok ? myrow / H : 0), myhead = row_ok ? myrow % H : 0;
  const int mylen = row_ok ? row_len[mytok] : 0;
  const int mylo = window > 0 ? max(0, mylen - window) : 0;
  const int maxlen = row_len[tok0 + ntok - 1];
  const int kbase = window > 0 ? (max(0, row_len[tok0] - window) / DKT) * DKT : 0;
  const int nsplit = gridDim.y;
  if (nsplit > 1) {
    if ((int)blockIdx.y >= ranges_used(longest, nsplit, split_keys, least_keys(longest))) return;
    split_keys = range_keys(longest, nsplit, split_keys, least_keys(longest));
  }
  const int kbeg = nsplit > 1 ? kbase + blockIdx.y * split_keys : kbase;
  const int kend = nsplit > 1 ? min(maxlen, kbeg + split_keys) : maxlen;
  const int* bt = tables + (int64_t)seq * W;
  const float scale2 = scale * LOG2E;

  Tile tf;
  if (kbeg < kend) tf.load(cache, bt, bs, Dk, kbeg, kend);
  bf16x8_t qf[NKS];
  const bf16_t* qr = q_abs + ((int64_t)mytok * H + myhead) * Dk;
  const bool vec = (Dk & 7) == 0;
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int d0 = ks * 32 + kq * 8;
    u32x4_t t = {0, 0, 0, 0};
    if (row_ok && d0 < Dk) {
      if (vec) {
        t = *reinterpret_cast<const u32x4_t*>(qr + d0);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (d0 + i < Dk) t[i >> 1] |= (uint32_t)qr[d0 + i] << (16 * (i & 1));
      }
    }
    qf[ks] = __builtin_bit_cast(bf16x8_t, t);
  }
  f32x4_t o[NCW];
#pragma unroll
  for (int n = 0; n < NCW; ++n) o[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const bf16_t* const vcol = sK + (4 * kq + (r16 >> 2)) * KS + 4 * (r16 & 3) + wave * 16 * NCW;
  for (int k0 = kbeg; k0 < kend; k0 += DKT) {
    __syncthreads();  // the previous tile is no longer read
    tf.store(sK);
    __syncthreads();
    if (k0 + DKT < kend) tf.load(cache, bt, bs, Dk, k0 + DKT, kend);
    f32x4_t a = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const bf16x8_t ka = *reinterpret_cast<const bf16x8_t*>(&sK[(wave * 16 + r16) * KS + ks * 32 + kq * 8]);
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qf[ks], a, 0, 0, 0);
    }
    float4 s4;
    float* const sp = &s4.x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = k0 + wave * 16 + kq * 4 + r;
      sp[r] = ((key < min(mylen, kend)) & (key >= mylo)) ? a[r] * scale2 : -INFINITY;
    }
    *reinterpret_cast<float4*>(&sS[r16 * SS + wave * 16 + kq * 4]) = s4;
    __syncthreads();
    // the row's 64 scores over four lanes: keys 32 t + 4 kq .. + 3 and 32 t + 16 + 4 kq .. + 3
    float p[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = *reinterpret_cast<const float4*>(&sS[r16 * SS + i * 16 + kq * 4]);
      p[4 * i] = v.x;
      p[4 * i + 1] = v.y;
      p[4 * i + 2] = v.z;
      p[4 * i + 3] = v.w;
    }
    float mx = p[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, p[i]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const float mref = (mn == -INFINITY) ? 0.f : mn;
    const float corr = __builtin_amdgcn_exp2f(m - mref);
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p[i] = __builtin_amdgcn_exp2f(p[i] - mref);
      psum += p[i];
    }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l = l * corr + psum;
    m = mn;
    float cr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) cr[r] = __shfl(corr, kq * 4 + r, 64);
    bf16x8_t ph[2], pl[2];
    split_weights(p, ph[0], pl[0]);
    split_weights(p + 8, ph[1], pl[1]);
#pragma unroll
    for (int n = 0; n < NCW; ++n) {
      f32x4_t acc = o[n];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] *= cr[r];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16x8_t vb = column_keys<KS>(vcol + t * 32 * KS + n * 16);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph[t], vb, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[t], vb, acc, 0, 0, 0);
      }
      o[n] = acc;
    }
  }
  // o[n][r] = O[row0 + 4 kq + r][column 16 (NCW wave + n) + r16]
  if (nsplit > 1) {
    const int64_t pbase = ((int64_t)blockIdx.x * nsplit + blockIdx.y) * 64 + row0;
    if (wave == 0 && kq == 0) {
      part_ml[(pbase + r16) * 2] = m;
      part_ml[(pbase + r16) * 2 + 1] = l;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int n = 0; n < NCW; ++n) {
        const int col = (wave * NCW + n) * 16 + r16;
        if (col < R) part_o[(pbase + kq * 4 + r) * R + col] = o[n][r];
      }
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float w = 1.f / __shfl(l, kq * 4 + r, 64);
    const int row = row0 + kq * 4 + r;
    if (row >= ntok * H) continue;
    const int64_t base = ((int64_t)(tok0 + row / H) * H + row % H) * R;
    if (gate) w *= 1.f / (1.f + expf(-ld(gate + (int64_t)(tok0 + row / H) * gate_stride + row % H)));
#pragma unroll
    for (int n = 0; n < NCW; ++n) {
      const int col = (wave * NCW + n) * 16 + r16;
      if (col < R) st(out + base + col, o[n][r] * w);
    }
  }
}

// Merge the key-range partials of a split step: out = sum_y 2^(m_y - M) o_y / sum_y 2^(m_y - M) l_y.
__global__ __launch_bounds__(NT) void latent_attention_merge_kernel(const int* __restrict__ items, int nsplit,
                                                                   const float* __restrict__ part_o,
                                                                   const float* __restrict__ part_ml, int H, int R,
                                                                   bf16_t* __restrict__ out,
                                                                   const bf16_t* __restrict__ gate,
                                                                   int64_t gate_stride, int split_keys,
                                                                   const int* __restrict__ longest) {
  const int item = blockIdx.x, row = blockIdx.y;
  const int tok0 = items[item * 3 + 1], ntok = items[item * 3 + 2];
  if (row >= ntok * H) return;
  const int64_t p0 = (int64_t)item * nsplit * 64 + row;
  const int64_t tok = tok0 + row / H, h = row % H;
  const float w = gate ? 1.f / (1.f + expf(-ld(gate + tok * gate_stride + h))) : 1.f;
  merge_ranges<NT>(part_ml + p0 * 2, 128, part_o + p0 * R, (int64_t)64 * R, ranges_used(longest, nsplit, split_keys, least_keys(longest)), R,
                   [](float x) { return exp2f(x); }, [&](int c, float v) { st(out + (tok * H + h) * R + c, v * w); });
}

template <typename T, int RC>
int launch_attn(const void* q_abs, const void* cache, const int* tables, int W, int bs, const int* row_seq,
                const int* row_len, float scale, int H, int R, int Dk, int T_rows, int QT, void* out,
                const void* gate, int64_t gate_stride, int window, hipStream_t stream) {
  // key tile: as many of 64 / 32 / 16 rows as fit beside the queries in 128 KB of LDS
  int KT = 64;
  while (KT > 16 && ((size_t)KT * (Dk + 1) + (size_t)QT * 4 * Dk) * 4 > 128 * 1024) KT >>= 1;
  const size_t lds = ((size_t)KT * (Dk + 1) + (size_t)QT * 4 * Dk) * 4;
  if (lds > 160 * 1024) return 1;
  const dim3 grid((T_rows + QT - 1) / QT, (H + 3) / 4);
  auto go = [&](auto kern) {
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, grid, dim3(NT), lds, stream, (const T*)q_abs, (const T*)cache, tables, W, bs, row_seq,
                       row_len, scale, H, R, Dk, KT, T_rows, (T*)out, (const T*)gate, gate_stride, window);
  };
  if (QT == 4) go(latent_attention_kernel<T, RC, 4>);
  else go(latent_attention_kernel<T, RC, 1>);
  return 0;
}

// out[t][h][n] = sum_k x[t][h][k] W[h][n][k] of a few rows t: a latent layer's ways into the latent space and back in a step of single
// tokens, each row of W what one number multiplies. A stream over W (2 MB at 16 heads) and a launch: a workgroup takes 16 rows of a head's W, its four
// waves a quarter of k each, 16 bytes per lane straight from memory with x beside them, and the quarters meet in LDS.
// us, torch.bmm / here: 16 heads, 512 -> 128 10.1 / 3.9 at one row, 10.2 / 4.1 at 9, 9.1 / 5.6 at 64; 128 -> 512 4.5 / 3.0 at 9, 4.8 / 4.3 at 64.
// Every workgroup of a head reads all of its x: 128 heads 9.5 / 8.0 at 16 rows, 9.5 / 11.8 at 32, 64 heads 9.2 / 5.8 at 32, 9.5 / 10.7 at 64,
// hence up to 2048 rows of heads.
template <int MB>
__global__ __launch_bounds__(NT) void head_product_kernel(const bf16_t* __restrict__ x, int64_t xt, int64_t xh,
                                                          const bf16_t* __restrict__ w, int K, int N, int T,
                                                          bf16_t* __restrict__ out, int64_t ot, int64_t oh) {
  __shared__ __attribute__((aligned(16))) f32x4_t red[3][MB][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
  const int h = blockIdx.y, n0 = blockIdx.x * 16, kw = K / 4;
  const bf16_t* wp = w + ((int64_t)h * N + n0 + c16) * K + wave * kw + 8 * g;
  const bf16_t* xp[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) xp[b] = x + min(16 * b + c16, T - 1) * xt + h * xh + wave * kw + 8 * g;
  f32x4_t acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < kw; k += 32) {
    const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(wp + k);
#pragma unroll
    for (int b = 0; b < MB; ++b)
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, *reinterpret_cast<const bf16x8_t*>(xp[b] + k), acc[b], 0, 0, 0);
  }
  if (wave > 0)
#pragma unroll
    for (int b = 0; b < MB; ++b) red[wave - 1][b][lane] = acc[b];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const f32x4_t v = (acc[b] + red[0][b][lane]) + (red[1][b][lane] + red[2][b][lane]);
    const int t = 16 * b + c16;
    if (t >= T) continue;
    bf16_t* o = out + t * ot + h * oh + n0 + 4 * g;
#pragma unroll
    for (int e = 0; e < 4; ++e) st(o + e, v[e]);
  }
}

}  // namespace

extern "C" {

// W [H][N][K]; x and out: rows of heads at xt, xh and ot, oh elements. -1: not on these operands
int sm_head_product(const void* x, int64_t xt, int64_t xh, const void* w, int H, int K, int N, int T, void* out, int64_t ot,
                    int64_t oh, hipStream_t stream) {
  if (T == 0 || H == 0 || N == 0) return 0;
  if (T > 64 || (int64_t)T * H > 2048 || K < 128 || K % 128 || N % 16 || H > 65535 || (((uintptr_t)w | (uintptr_t)x) & 15) || xt % 8 || xh % 8) return -1;
  const dim3 grid(N / 16, H);
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, stream, (const bf16_t*)x, xt, xh, (const bf16_t*)w, K, N, T, (bf16_t*)out, ot, oh);
  };
  if (T <= 16) go(head_product_kernel<1>);
  else if (T <= 32) go(head_product_kernel<2>);
  else if (T <= 48) go(head_product_kernel<3>);
  else go(head_product_kernel<4>);
  return 0;
}

void sm_latent_rope_cache(const void* q, int64_t q_stride, const void* kv, int64_t kv_stride, const void* norm_w,
                          float eps, const int64_t* positions, const float* cos_sin, int H, int dn, int dr,
                          int rot_dims, int R, const int64_t* slots, void* cache, void* q_abs, int interleaved, int T,
                          int f32, hipStream_t stream) {
  if (T == 0) return;
  if (f32)
    hipLaunchKernelGGL((latent_rope_cache_kernel<float>), dim3(T), dim3(NT), 0, stream, (const float*)q, q_stride,
                       (const float*)kv, kv_stride, (const float*)norm_w, eps, positions, cos_sin, H, dn, dr,
                       rot_dims, R, slots, (float*)cache, (float*)q_abs, interleaved);
  else
    hipLaunchKernelGGL((latent_rope_cache_kernel<bf16_t>), dim3(T), dim3(NT), 0, stream, (const bf16_t*)q, q_stride,
                       (const bf16_t*)kv, kv_stride, (const bf16_t*)norm_w, eps, positions, cos_sin, H, dn, dr,
                       rot_dims, R, slots, (bf16_t*)cache, (bf16_t*)q_abs, interleaved);
}

// Latents and rotated parts of sequences first .. first + n - 1, at most ``longest`` keys each.
void sm_latent_gather(const void* cache, const int* tables, int W, int bs, const int* base, int first, int n, int longest, int R, int dr,
                      void* lat, void* rot, hipStream_t stream) {
  if (n == 0 || longest == 0) return;
  hipLaunchKernelGGL(latent_gather_kernel, dim3((unsigned)(((int64_t)longest * ((R + dr) / 8) + NT - 1) / NT), n), dim3(NT), 0, stream,
                     (const bf16_t*)cache, tables, W, bs, base, first, R, dr, (bf16_t*)lat, (bf16_t*)rot);
}

// q [T, H, 128 + 64] rows q_stride apart, of which the first 128; the rotated 64 at q_rot + row * rot_stride + head * rot_head; items of up
// to 64 tokens; kv [keys, H, 128 + 128], rot [keys, 64] of the gathered sequences; out [T, H, 128] (rows of the items), tokens out_stride apart:
// H heads of more may be asked for.
void sm_latent_own(const void* q, int64_t q_stride, const void* q_rot, int64_t rot_stride, int64_t rot_head, const void* kv, const void* rot,
                   const int* base, const int* items, int n_items, const int* row_len, float scale, int H, void* out, int64_t out_stride,
                   const void* gate, int64_t gate_stride, hipStream_t stream) {
  if (n_items == 0) return;
  hipLaunchKernelGGL(latent_own_kernel, dim3(H, n_items), dim3(NT), 0, stream, (const bf16_t*)q, q_stride, (const bf16_t*)q_rot, rot_stride,
                     rot_head, (const bf16_t*)kv, (const bf16_t*)rot, base, items, row_len, scale, H, (bf16_t*)out, out_stride,
                     (const bf16_t*)gate, gate_stride);
}

// Returns 0, or 1 when the sizes do not fit the kernel (R > 1024 or rows too wide for LDS).
int sm_latent_attention(const void* q_abs, const void* cache, const int* tables, int W, int bs, const int* row_seq,
                        const int* row_len, float scale, int H, int R, int Dk, int T, int QT, void* out, int f32,
                        const void* gate, int64_t gate_stride, int window, hipStream_t stream) {
  if (T == 0) return 0;
  const int rc = (R + 63) / 64;
#define SM_GO(TYPE, RC) return launch_attn<TYPE, RC>(q_abs, cache, tables, W, bs, row_seq, row_len, scale, H, R, Dk, T, QT, out, gate, gate_stride, window, stream)
  if (f32) {
    if (rc <= 1) SM_GO(float, 1);
    if (rc <= 2) SM_GO(float, 2);
    if (rc <= 4) SM_GO(float, 4);
    if (rc <= 8) SM_GO(float, 8);
    if (rc <= 16) SM_GO(float, 16);
  } else {
    if (rc <= 1) SM_GO(bf16_t, 1);
    if (rc <= 2) SM_GO(bf16_t, 2);
    if (rc <= 4) SM_GO(bf16_t, 4);
    if (rc <= 8) SM_GO(bf16_t, 8);
    if (rc <= 16) SM_GO(bf16_t, 16);
  }
#undef SM_GO
  return 1;
}

// bf16, matrix cores. items [n, 3] = (sequence, first token row, tokens), tokens * H <= 64.
// rows > 0: a step of single tokens whose items have at most ``rows`` rows; the waves share an item.
// nsplit > 1: every item's keys are cut into nsplit ranges of split_keys (a multiple of 32, of 64 with
// rows > 0) that run as separate workgroups; part_o [n * nsplit * 64 * R] and part_ml [n * nsplit * 64 * 2]
// fp32 hold their partial results and a second kernel merges them.
// longest: null, or the step's longest context on the device, which then sizes the ranges (range_keys).
// Returns 0, or 1 when the sizes are outside the compiled forms (Dk > 576, R > 512, H > 64).
int sm_latent_attention_mfma(const void* q_abs, const void* cache, const int* tables, int W, int bs, const int* items,
                             int n_items, const int* row_len, float scale, int H, int R, int Dk, void* out,
                             int nsplit, int split_keys, float* part_o, float* part_ml, const void* gate,
                             int64_t gate_stride, int window, int rows, const int* longest,
                             hipStream_t stream) {
  if (n_items == 0) return 0;
  const int nks = (Dk + 31) / 32, ncb = (R + 15) / 16;
  if (H > 64 || nks > 18 || ncb > 32) return 1;
  if (rows == 0 && nsplit == 1 && (Dk == 512 || Dk == 576) && bs % MKT == 0 &&
      (((uintptr_t)q_abs | (uintptr_t)cache | (uintptr_t)out) & 15) == 0) {
#define SM_GO(NKS)                                                                                                   \
  hipLaunchKernelGGL(latent_prompt_kernel<NKS>, dim3(n_items), dim3(NT), 0, stream, (const bf16_t*)q_abs,            \
                     (const bf16_t*)cache, tables, W, bs, items, row_len, scale, H, R, (bf16_t*)out,                 \
                     (const bf16_t*)gate, gate_stride, window)
    if (Dk == 512) SM_GO(16);
    else SM_GO(18);
#undef SM_GO
    return 0;
  }
  const dim3 grid(n_items, nsplit, rows > 0 ? (rows + 15) / 16 : 1);
#define SM_GO2(KERN)                                                                                                 \
  hipLaunchKernelGGL((KERN), grid, dim3(NT), 0, stream, (const bf16_t*)q_abs, (const bf16_t*)cache, tables, W, bs,   \
                     items, row_len, scale, H, R, Dk, (bf16_t*)out, split_keys, part_o, part_ml,                     \
                     nsplit > 1 ? nullptr : (const bf16_t*)gate, gate_stride, window, longest)
#define SM_GO(NKS, NCB)                                                            \
  do {                                                                             \
    if (rows > 0) SM_GO2((latent_decode_mfma_kernel<NKS, NCB / 4>));               \
    else SM_GO2((latent_attention_mfma_kernel<NKS, NCB>));                         \
  } while (0)
  if (nks <= 2 && ncb <= 4) SM_GO(2, 4);
  else if (nks <= 4 && ncb <= 8) SM_GO(4, 8);
  else if (nks <= 6 && ncb <= 8) SM_GO(6, 8);
  else if (nks <= 8 && ncb <= 16) SM_GO(8, 16);
  else if (nks <= 10 && ncb <= 16) SM_GO(10, 16);
  else if (nks <= 16 && ncb <= 32) SM_GO(16, 32);
  else SM_GO(18, 32);
#undef SM_GO
#undef SM_GO2
  if (nsplit > 1)
    hipLaunchKernelGGL(latent_attention_merge_kernel, dim3(n_items, rows > 0 ? rows : 64), dim3(NT), 0, stream, items,
                       nsplit, part_o, part_ml, H, R, (bf16_t*)out, (const bf16_t*)gate, gate_stride, split_keys, longest);
  return 0;
}

}  // extern "C"
