// Gated delta rule over a step's per-sequence token runs (seq_start [n+1]), each continuing the
// state in its slot (seq_slot) or starting from zero (seq_init == 0). The state S [dk, dv] per head
// is fp32.
//
//   q, k <- unit vectors (x / sqrt(sum x^2 + 1e-6)), q times dk^-1/2
//   g = exp(-A_h softplus(a + dt_bias))   one per head, or one per head and key channel (row of S)
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//   out = o / rms(o) * norm_w * gate,  gate = silu or sigmoid of its input
//
// Only the recurrence is sequential, so it is all the scan kernel does. A first kernel, parallel
// over the tokens, makes the unit queries and keys, the decays and beta (fp32, rows padded to
// KD = 32 .. 256 with q = k = 0 and g = 1); a last one, parallel again, norms the read-outs and applies
// the gate. The columns of S never meet in the recurrence, so the scan has no barrier: a workgroup
// is ONE wave that owns 16 (or 8) value columns of one head and sequence, lane = (column c, row group
// r of 4 (or 8)), and keeps rows [r KR, (r + 1) KR) of its column in registers. The two sums over the
// key rows (S^T k and S^T q) end with DPP exchanges between the lanes of a column. The key-side
// vectors reach the wave in blocks of tokens through LDS, fetched a block ahead. Steps with few
// (head, sequence) pairs - a prompt - take the 8 x 8 form: twice the waves, half the work of each.
#include "seqmix_common.h"
#include <algorithm>

using namespace sm;

namespace {

constexpr int NT = 256;

// Unit queries and keys, decays and beta of every token (fp32). qn, kn [T, G, KD]; dec [T, H, KD]
// (one decay per key channel) or [T, H]; beta [T, H]. Rows beyond dk: q = k = 0, g = 1.
template <typename T>
__global__ __launch_bounds__(NT) void delta_prep_kernel(const T* __restrict__ xc, int64_t x_stride, int G, int dk,
                                                       int KD, int H, const T* __restrict__ beta_raw,
                                                       int64_t beta_stride, const T* __restrict__ decay_raw,
                                                       int64_t decay_stride, int per_channel,
                                                       const float* __restrict__ A, const float* __restrict__ dt_bias,
                                                       float* __restrict__ qn, float* __restrict__ kn,
                                                       float* __restrict__ dec, float* __restrict__ beta) {
  const int64_t t = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const T* xr = xc + t * x_stride;
  const float qscale = 1.f / sqrtf((float)dk);
  for (int hd = wave; hd < 2 * G; hd += NT / 64) {  // q heads, then k heads: back to back in the row
    float r[4], ss = 0.f;                           // KD <= 256
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = lane + 64 * i;
      r[i] = e < dk ? ld(xr + hd * dk + e) : 0.f;
      ss += r[i] * r[i];
    }
    const float inv = Fn<T>::rsqrt(wave_sum(ss) + 1e-6f) * (hd < G ? qscale : 1.f);
    float* dst = (hd < G ? qn + (t * G + hd) * KD : kn + (t * G + hd - G) * KD);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = lane + 64 * i;
      if (e < KD) dst[e] = r[i] * inv;
    }
  }
  if (per_channel) {
    for (int idx = threadIdx.x; idx < H * KD; idx += NT) {
      const int h = idx / KD, i = idx - h * KD;
      float g = 1.f;
      if (i < dk) g = Fn<T>::exp(-A[h] * Fn<T>::softplus(ld(decay_raw + t * decay_stride + h * dk + i) + dt_bias[h * dk + i]));
      dec[t * H * KD + idx] = g;
    }
  }
  for (int h = threadIdx.x; h < H; h += NT) {
    if (!per_channel) dec[t * H + h] = Fn<T>::exp(-A[h] * Fn<T>::softplus(ld(decay_raw + t * decay_stride + h) + dt_bias[h]));
    beta[t * H + h] = Fn<T>::sigmoid(ld(beta_raw + t * beta_stride + h));
  }
}

// HGRN2: queries, gates and write strengths of every token (fp32), from the projection [q | f | ...].
// qn = silu(q), dec = f = lower + (1 - lower) sigmoid(f_raw + bias), kn = 1 - f; all [T, H, KD].
// Rows beyond dk: q = k = 0, f = 1.
template <typename T>
__global__ __launch_bounds__(NT) void hgrn2_prep_kernel(const T* __restrict__ p, int64_t p_stride, int H, int dk,
                                                       int KD, const float* __restrict__ f_bias,
                                                       const float* __restrict__ lower, float* __restrict__ qn,
                                                       float* __restrict__ kn, float* __restrict__ dec) {
  const int64_t t = blockIdx.x;
  const T* pr = p + t * p_stride;
  for (int idx = blockIdx.y * NT + threadIdx.x; idx < H * KD; idx += gridDim.y * NT) {
    const int h = idx / KD, i = idx - h * KD;
    float q = 0.f, k = 0.f, f = 1.f;
    if (i < dk) {
      const int c = h * dk + i;
      q = Fn<T>::silu(ld(pr + c));
      const float lo = lower[c];
      const float sg = Fn<T>::sigmoid(ld(pr + H * dk + c) + f_bias[c]);
      f = lo + (1.f - lo) * sg;
      k = (1.f - lo) * (1.f - sg);  // 1 - f without the cancellation near f = 1
    }
    qn[t * H * KD + idx] = q;
    kn[t * H * KD + idx] = k;
    dec[t * H * KD + idx] = f;
  }
}

// Sum over the RG (4 or 8) neighbouring lanes of a column (lanes RG c .. RG c + RG - 1): DPP
// exchanges, no LDS. After the two quad exchanges all four lanes of a quad hold the quad's sum; the
// mirror inside a half row (lane i <-> 7 - i) then brings the other quad's.
template <int RG>
__device__ __forceinline__ float group_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));  // 1 0 3 2
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));  // 2 3 0 1
  if (RG == 8)
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));  // half mirror
  return v;
}

// The recurrence. One wave per (head, block of 64 / RG value columns, sequence); RG = 4 or 8 row groups
// (lanes) per column, KR rows per lane. CH: a decay per key row.
// The key-side vectors of TB tokens at a time go through LDS: while the wave computes one block of
// tokens from one buffer, the next block's loads are in flight into registers, and are written to the
// other buffer afterwards - the recurrence never waits for global memory. Per token a lane reads its
// KR rows of k, q (and g) as 16-byte LDS broadcasts.
// OUT = false: the state alone is advanced (no read-out) - the first pass of the chunked form below.
template <typename T, int KR, int RG, bool CH, int TB, bool DELTA = true, bool OUT = true>
__global__ __launch_bounds__(64) void gated_delta_scan_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn, const float* __restrict__ dec,
    const float* __restrict__ beta, const T* __restrict__ xc, int64_t x_stride, int voff, int G, int dk, int H, int dv,
    float* __restrict__ state, const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_init, float* __restrict__ o_raw, float* __restrict__ run_decay = nullptr) {
  constexpr int KD = RG * KR, CPW = 64 / RG, NV = CH ? 3 : 2;       // vectors per token: k, q (, g)
  constexpr int C4 = KD / 4;                         // 16-byte chunks per vector
  constexpr int NL = TB * NV * C4 / 64;              // chunks per lane and block (KD >= 32: a whole number)
  __shared__ __attribute__((aligned(16))) float buf[2][TB * NV * KD];
  const int ncb = (dv + CPW - 1) / CPW;
  const int h = blockIdx.x / ncb, cb = blockIdx.x - h * ncb, s = blockIdx.y;
  const int lane = threadIdx.x, r = lane % RG, c = lane / RG;
  const int col = cb * CPW + c;
  const bool colok = col < dv;
  const int qh = h / (H / G);
  const int row0 = r * KR;
  const int lo = seq_start[s], hi = seq_start[s + 1];
  if (lo >= hi) return;
  float* sp = state + ((int64_t)seq_slot[s] * H + h) * dk * dv;
  const bool init = seq_init[s] != 0;
  float S[KR];
#pragma unroll
  for (int i = 0; i < KR; ++i) S[i] = (init && colok && row0 + i < dk) ? sp[(int64_t)(row0 + i) * dv + col] : 0.f;
  // pass 1 of the chunked form: the waves of a head's first column block also multiply the run's decays
  const bool want_decay = !OUT && CH && run_decay != nullptr && cb == 0;
  float D[(!OUT && CH) ? KR : 1];
#pragma unroll
  for (int i = 0; i < ((!OUT && CH) ? KR : 1); ++i) D[i] = 1.f;
  // one token: kp, qp, gp point at this lane's KR rows of k, q and (CH) g; returns the read-out
  auto token = [&](const float4* kp, const float4* qp, const float4* gp, float gj, float bj, float vj) {
    float k[KR];
    float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KR; i += 4) {
      const float4 k4 = kp[i >> 2];
      k[i] = k4.x; k[i + 1] = k4.y; k[i + 2] = k4.z; k[i + 3] = k4.w;
      if (CH) {
        const float4 g4 = gp[i >> 2];
        S[i] *= g4.x; S[i + 1] *= g4.y; S[i + 2] *= g4.z; S[i + 3] *= g4.w;
        if (!OUT && want_decay) {
          D[i] *= g4.x; D[i + 1] *= g4.y; D[i + 2] *= g4.z; D[i + 3] *= g4.w;
        }
      } else {
        S[i] *= gj; S[i + 1] *= gj; S[i + 2] *= gj; S[i + 3] *= gj;
      }
      if (DELTA) {
        p[0] += k[i] * S[i];
        p[1] += k[i + 1] * S[i + 1];
        p[2] += k[i + 2] * S[i + 2];
        p[3] += k[i + 3] * S[i + 3];
      }
    }
    const float pred = DELTA ? group_sum<RG>((p[0] + p[1]) + (p[2] + p[3])) : 0.f;
    const float u = DELTA ? bj * (vj - pred) : vj;
    float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KR; i += 4) {
      const float4 q4 = qp[i >> 2];
      S[i] += k[i] * u; S[i + 1] += k[i + 1] * u; S[i + 2] += k[i + 2] * u; S[i + 3] += k[i + 3] * u;
      if (OUT) {
        o[0] += S[i] * q4.x;
        o[1] += S[i + 1] * q4.y;
        o[2] += S[i + 2] * q4.z;
        o[3] += S[i + 3] * q4.w;
      }
    }
    return OUT ? group_sum<RG>((o[0] + o[1]) + (o[2] + o[3])) : 0.f;
  };
  if (hi - lo <= 2) {
    // a decoded token (or two): the lane's rows straight from global memory, no staging
    for (int64_t t = lo; t < hi; ++t) {
      const float4* kp = reinterpret_cast<const float4*>(kn + (t * G + qh) * KD + row0);
      const float4* qp = reinterpret_cast<const float4*>(qn + (t * G + qh) * KD + row0);
      const float4* gp = reinterpret_cast<const float4*>(CH ? dec + (t * H + h) * KD + row0 : kn);
      const float vj = colok ? ld(xc + t * x_stride + voff + h * dv + col) : 0.f;
      const float ov = token(kp, qp, gp, CH ? 1.f : dec[t * H + h], DELTA ? beta[t * H + h] : 1.f, vj);
      if (OUT && r == 0 && colok) o_raw[t * H * dv + h * dv + col] = ov;
    }
  } else {
    float4 stage[NL];
    float vb[TB], bb[TB], gb[CH ? 1 : TB];            // the block's values, betas and per-head decays
    auto fetch = [&](int t0) {                          // block t0 .. t0 + TB - 1 -> registers
#pragma unroll
      for (int n = 0; n < NL; ++n) {
        const int e = lane + 64 * n;
        const int j = e / (NV * C4), rem = e - j * (NV * C4);
        const int var = rem / C4, i4 = rem - var * C4;
        const int64_t t = t0 + j;
        float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < hi) {
          const float* src =
              var == 0 ? kn + (t * G + qh) * KD : var == 1 ? qn + (t * G + qh) * KD : dec + (t * H + h) * KD;
          v4 = reinterpret_cast<const float4*>(src)[i4];
        }
        stage[n] = v4;
      }
#pragma unroll
      for (int j = 0; j < TB; ++j) {
        const int64_t t = t0 + j;
        vb[j] = bb[j] = 0.f;
        if (!CH) gb[j] = 1.f;
        if (t >= hi) continue;
        vb[j] = colok ? ld(xc + t * x_stride + voff + h * dv + col) : 0.f;
        bb[j] = DELTA ? beta[t * H + h] : 1.f;
        if (!CH) gb[j] = dec[t * H + h];
      }
    };
    auto spill = [&](int which) {                       // registers -> LDS buffer
#pragma unroll
      for (int n = 0; n < NL; ++n) reinterpret_cast<float4*>(buf[which])[lane + 64 * n] = stage[n];
    };
    fetch(lo);
    spill(0);
    __syncthreads();
    int which = 0;
    for (int t0 = lo; t0 < hi; t0 += TB, which ^= 1) {
      float cv[TB], cbeta[TB], cg[CH ? 1 : TB];
#pragma unroll
      for (int j = 0; j < TB; ++j) {
        cv[j] = vb[j];
        cbeta[j] = bb[j];
        if (!CH) cg[j] = gb[j];
      }
      const bool more = t0 + TB < hi;
      if (more) fetch(t0 + TB);
      const float* bk = buf[which];
#pragma unroll
      for (int j = 0; j < TB; ++j) {
        if (t0 + j >= hi) break;
        const float ov = token(reinterpret_cast<const float4*>(bk + (j * NV + 0) * KD + row0),
                               reinterpret_cast<const float4*>(bk + (j * NV + 1) * KD + row0),
                               reinterpret_cast<const float4*>(bk + (j * NV + (CH ? 2 : 0)) * KD + row0),
                               CH ? 1.f : cg[j], cbeta[j], cv[j]);
        if (OUT && r == 0 && colok) o_raw[(int64_t)(t0 + j) * H * dv + h * dv + col] = ov;
      }
      if (more) spill(which ^ 1);
      __syncthreads();  // one wave: orders the buffer's writes before the next block's reads
    }
  }
  if (colok) {
#pragma unroll
    for (int i = 0; i < KR; ++i)
      if (row0 + i < dk) sp[(int64_t)(row0 + i) * dv + col] = S[i];
  }
  if (!OUT && CH && want_decay && c == 0) {
#pragma unroll
    for (int i = 0; i < KR; ++i) run_decay[((int64_t)s * H + h) * KD + row0 + i] = D[i];
  }
}

// Chunked form of the recurrence without the delta term, for prompts in float32 or of heads above 128 (otherwise the
// matrix-core form below): S <- diag(g) S + k v^T is linear in
// S, so a run cut into chunks can be scanned in all chunks at once. Pass 1 scans every chunk from zero
// (its own contribution L_c, no read-out) and multiplies the chunk's decays (D_c, one per key row); the
// small kernel below walks a sequence's chunks in order, S_(c+1) = D_c S_c + L_c, leaving every
// chunk's true start state where its L_c was and the run's final state in the sequence's slot; pass 2
// scans every chunk again from its start state and reads out. All fp32; against the token-by-token scan
// only the order of the additions that form a chunk's start state differs.
// c_state [chunks, H, dk, dv]: in L_c, out the start state of chunk c. s_chunk0 [nseq + 1] bounds each
// sequence's chunks.
__global__ __launch_bounds__(NT) void chunk_link_kernel(float* __restrict__ c_state, const float* __restrict__ c_decay,
                                                       const int* __restrict__ s_chunk0, int H, int dk, int dv, int KD,
                                                       float* __restrict__ state, const int* __restrict__ seq_slot,
                                                       const int* __restrict__ seq_init) {
  const int s = blockIdx.y;
  const int64_t n = (int64_t)H * dk * dv;
  const int c0 = s_chunk0[s], c1 = s_chunk0[s + 1];
  if (c0 >= c1) return;
  float* sp = state + (int64_t)seq_slot[s] * n;
  const bool init = seq_init[s] != 0;
  for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < n; e += (int64_t)gridDim.x * NT) {
    const int h = (int)(e / ((int64_t)dk * dv)), i = (int)((e / dv) % dk);
    float S = init ? sp[e] : 0.f;
    for (int c = c0; c < c1; ++c) {
      const float own = c_state[(int64_t)c * n + e];
      c_state[(int64_t)c * n + e] = S;
      S = c_decay[((int64_t)c * H + h) * KD + i] * S + own;
    }
    sp[e] = S;
  }
}

// out = o / rms(o) * norm_w * gate per head; a wave per (token, head), any dv.
template <typename T>
__global__ __launch_bounds__(NT) void delta_out_kernel(const float* __restrict__ o_raw, const T* __restrict__ gate_raw,
                                                      int64_t gate_stride, int gate_sigmoid,
                                                      const T* __restrict__ norm_w, float eps, int H, int dv,
                                                      T* __restrict__ out) {
  const int64_t t = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int h = blockIdx.y * (NT / 64) + wave; h < H; h += gridDim.y * (NT / 64)) {
    const float* orow = o_raw + (t * H + h) * dv;
    float ss = 0.f;
    for (int e = lane; e < dv; e += 64) ss += orow[e] * orow[e];
    const float inv = Fn<T>::rsqrt(wave_sum(ss) / (float)dv + eps);
    for (int e = lane; e < dv; e += 64) {
      float gt = 1.f;  // no gate: the norm alone
      if (gate_raw != nullptr) {
        const float gr = ld(gate_raw + t * gate_stride + h * dv + e);
        gt = gate_sigmoid ? Fn<T>::sigmoid(gr) : Fn<T>::silu(gr);
      }
      st(out + (t * H + h) * dv + e, orow[e] * inv * ld(norm_w + e) * gt);
    }
  }
}

// ---- HGRN2 over prompts, on the matrix cores (fp32). Within a chunk of CT = 64 tokens the recurrence is an attention whose
// scores carry the decays between the two tokens per key row, A[t, s] = sum_i q_t,i k_s,i prod_{s < u <= t} f_u,i, and a chunk
// meets the earlier ones through the state it starts from. The products of decays are never divided (a decay may be as small
// as it likes): a pair of tokens is handled where its two places first part, at a boundary in multiples of h = 1, 2, 4 or 8
// tokens for two tokens of a block of 16, so both sides are products of factors on the way to that boundary,
//   q^_t = q_t prod_{boundary <= u <= t} f_u,   k^_s = k_s prod_{s < u < boundary} f_u.
// One 16 x 16 product per h gives all pairs of that h; a lane keeps the one that is its pair's. Both sides for twice the h
// are the old ones times the total of the neighbouring half block, one lane exchange. Blocks of 16 meet through
// the totals of the blocks between them. Every wave owns one block of 16 tokens: lane = (token r16, key rows
// 16 ks + 4 kq + j), which is the operand layout of the products, so scores never pass through LDS.
// Three kernels: every chunk's own contribution to the state with its total decay, the walk over a sequence's chunks, the
// read-outs with their norm. bf16 storage only: a sum of 64 products takes one rounding per product here and one per four
// products and lane in the scan above, which float32 results would show (1.1e-7 off in 64 bits against 1.0e-7).
// 2048 tokens, 32 heads x 64 x 64: 333 us with two scans of every chunk, now 72 us (21 + 11 + 40; the read-outs' matrix
// instructions take 14, their decays about as long).
constexpr int CT = 64, CS = CT + 4;  // chunk, LDS row stride of what is read along the tokens
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t load4(const float* p, int n, bool vec) {
  if (vec) return *reinterpret_cast<const f32x4_t*>(p);
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < n) v[j] = p[j];
  return v;
}
__device__ __forceinline__ f32x4_t load4(const bf16_t* p, int n, bool vec) {
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  if (vec) {
    const ushort4 b = *reinterpret_cast<const ushort4*>(p);
    v = f32x4_t{ld(&b.x), ld(&b.y), ld(&b.z), ld(&b.w)};
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < n) v[j] = ld(p + j);
  }
  return v;
}

// Decay f and write strength 1 - f of four key rows of a token (n of them are there).
__device__ __forceinline__ void gate4(const bf16_t* p, const float* f_bias, const float* lower, int n, bool vec, f32x4_t& f, f32x4_t& k) {
  const f32x4_t raw = load4(p, n, vec), b = load4(f_bias, n, vec), lo = load4(lower, n, vec);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float sg = Fn<bf16_t>::sigmoid(raw[j] + b[j]);
    f[j] = j < n ? lo[j] + (1.f - lo[j]) * sg : 1.f;
    k[j] = j < n ? (1.f - lo[j]) * (1.f - sg) : 0.f;  // 1 - f without the cancellation near f = 1
  }
}

// The value of the neighbouring group of HB lanes (of a row of 16), which is the same in all its lanes.
template <int HB>
__device__ __forceinline__ float other_half(float v) {
  constexpr int ctrl = HB == 1 ? 0xB1 : HB == 2 ? 0x4E : HB == 4 ? 0x141 : 0x140;  // quad permutes, half mirror, mirror
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true));
}
// From boundaries in multiples of HB tokens to 2 HB. total + rest = product of the decays of the lane's group of HB tokens:
// products of factors just below 1 all round the same way, which a slow key row would remember, so their roundings are kept.
struct Total {
  f32x4_t hi, lo;
  __device__ __forceinline__ void times(const f32x4_t h, const f32x4_t l) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p = hi[j] * h[j], r = __builtin_fmaf(hi[j], h[j], -p);
      lo[j] = __builtin_fmaf(lo[j], h[j], __builtin_fmaf(hi[j], l[j], r));
      hi[j] = p;
    }
  }
  __device__ __forceinline__ f32x4_t value() const { return hi + lo; }
};
template <int HB>
__device__ __forceinline__ f32x4_t widen(int r16, Total& total, f32x4_t& kh) {
  f32x4_t h, l, q;  // q: what the query side takes
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h[j] = other_half<HB>(total.hi[j]);
    l[j] = other_half<HB>(total.lo[j]);
    const float o = h[j] + l[j];
    kh[j] *= (r16 & HB) ? 1.f : o;
    q[j] = (r16 & HB) ? o : 1.f;
  }
  total.times(h, l);
  return q;
}

__device__ __forceinline__ f32x4_t mul_add4(const f32x4_t a, const f32x4_t b, f32x4_t c) {  // c + a b over 16 elements of K
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  return c;
}

// The chunk's values, transposed: vt[column][token], zeros past the chunk's end and past dv. Returns whether this lane's
// are all finite.
template <int NVT>
__device__ __forceinline__ bool stage_values(const bf16_t* row, bool there, int dv, bool vec, int kq, int tok, float* vt) {
  float zero = 0.f;
#pragma unroll
  for (int n = 0; n < NVT; ++n) {
    const int col = 16 * n + 4 * kq;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    if (there && col < dv) v = load4(row + col, dv - col, vec && col + 4 <= dv);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      vt[(col + j) * CS + tok] = v[j];
      zero = __builtin_fmaf(v[j], 0.f, zero);  // NaN from an infinity or a NaN
    }
  }
  return zero == 0.f;
}

// Every chunk's own state contribution, transposed ([dv][KD], KD = 16 NKS, zeros past dk), and the product of its decays [KD].
template <int NKS, int NVT>
__global__ __launch_bounds__(NT) void hgrn2_chunk_kernel(const bf16_t* __restrict__ p, int64_t p_stride, int H, int dk, int dv,
                                                        int vec, const float* __restrict__ f_bias,
                                                        const float* __restrict__ lower, const int* __restrict__ c_start,
                                                        int c_first, float* __restrict__ c_state,
                                                        float* __restrict__ c_decay) {
  constexpr int KD = 16 * NKS;
  __shared__ __attribute__((aligned(16))) float kt[KD * CS], vt[16 * NVT * CS], bt[8 * KD];  // bt: totals of the blocks, their rests
  const int h = blockIdx.x, c = c_first + blockIdx.y;
  const int t0 = c_start[c], n = min(c_start[c + 1] - t0, CT);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4, tok = 16 * wave + r16;
  const bool there = tok < n;
  const bf16_t* row = p + (int64_t)(t0 + (there ? tok : 0)) * p_stride;
  const bool any = 16 * wave < n;  // wave-uniform
  f32x4_t kh[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int i = 16 * ks + 4 * kq;
    Total total = {{1.f, 1.f, 1.f, 1.f}, {0.f, 0.f, 0.f, 0.f}};
    kh[ks] = total.lo;
    if (there && i < dk)
      gate4(row + (H + h) * dk + i, f_bias + h * dk + i, lower + h * dk + i, dk - i, vec != 0, total.hi, kh[ks]);
    if (any) {
      widen<1>(r16, total, kh[ks]);
      widen<2>(r16, total, kh[ks]);
      widen<4>(r16, total, kh[ks]);
      widen<8>(r16, total, kh[ks]);
    }
    if (r16 == 0) {
      *reinterpret_cast<f32x4_t*>(bt + wave * KD + i) = total.hi;
      *reinterpret_cast<f32x4_t*>(bt + (4 + wave) * KD + i) = total.lo;
    }
  }
  if (any) stage_values<NVT>(row + 2 * H * dk + h * dv, there, dv, vec != 0, kq, tok, vt);
  __syncthreads();
  auto block = [&](int b, int i) {
    return Total{*reinterpret_cast<const f32x4_t*>(bt + b * KD + i), *reinterpret_cast<const f32x4_t*>(bt + (4 + b) * KD + i)};
  };
  if (any) {
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int i = 16 * ks + 4 * kq;
      for (int b = wave + 1; b < 4; ++b) kh[ks] *= block(b, i).value();
#pragma unroll
      for (int j = 0; j < 4; ++j) kt[(i + j) * CS + tok] = kh[ks][j];
    }
  }
  for (int i = 4 * threadIdx.x; i < KD; i += 4 * NT) {
    Total d = block(0, i);
    for (int b = 1; b < 4; ++b) d.times(block(b, i).hi, block(b, i).lo);
    *reinterpret_cast<f32x4_t*>(c_decay + ((int64_t)c * H + h) * KD + i) = d.value();
  }
  __syncthreads();
  float* dst = c_state + ((int64_t)c * H + h) * dv * KD;
  const int nb = (n + 15) / 16;
  for (int e = wave; e < NKS * NVT; e += 4) {
    const int m = e / NKS, i = 16 * (e % NKS) + r16;
    if (16 * m >= dv) break;
    f32x4_t a = {0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < nb; ++b)
      a = mul_add4(*reinterpret_cast<const f32x4_t*>(vt + (16 * m + r16) * CS + 16 * b + 4 * kq),
                   *reinterpret_cast<const f32x4_t*>(kt + i * CS + 16 * b + 4 * kq), a);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (16 * m + 4 * kq + r < dv) dst[(16 * m + 4 * kq + r) * KD + i] = a[r];
  }
}

// c_state: in every chunk's own contribution, out the state it starts from (both transposed, [dv][KD]); the run's final state
// goes to the sequence's slot. Eight chunks' loads at a time: they do not wait for the walk.
__global__ __launch_bounds__(NT) void hgrn2_link_kernel(float* __restrict__ c_state, const float* __restrict__ c_decay,
                                                       const int* __restrict__ s_chunk0, int s_first, int H, int dk, int dv,
                                                       int KD, float* __restrict__ state,
                                                       const int* __restrict__ seq_slot,
                                                       const int* __restrict__ seq_init) {
  const int s = s_first + blockIdx.y, c0 = s_chunk0[s], c1 = s_chunk0[s + 1];
  const int64_t n = (int64_t)H * dv * KD, e = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (c0 >= c1 || e >= n) return;
  const int i = (int)(e % KD), col = (int)(e / KD % dv), h = (int)(e / ((int64_t)KD * dv));
  float* sp = state + (((int64_t)seq_slot[s] * H + h) * dk + i) * dv + col;
  float S = seq_init[s] != 0 && i < dk ? *sp : 0.f;
  float* own = c_state + e;
  const float* dec = c_decay + h * KD + i;
  for (int c = c0; c < c1; c += 8) {
    float a[8], d[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t cu = min(c + u, c1 - 1);
      a[u] = own[cu * n];
      d[u] = dec[cu * H * KD];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (c + u < c1) {
        own[(int64_t)(c + u) * n] = S;
        S = d[u] * S + a[u];
      }
  }
  if (i < dk) *sp = S;
}

template <int NKS, int NVT>
__global__ __launch_bounds__(NT) void hgrn2_read_kernel(const bf16_t* __restrict__ p, int64_t p_stride, int H, int dk, int dv, int vec,
                                                       const float* __restrict__ f_bias, const float* __restrict__ lower,
                                                       const int* __restrict__ c_start, int c_first, const float* __restrict__ c_state,
                                                       const bf16_t* __restrict__ norm_w, float eps, bf16_t* __restrict__ out) {
  constexpr int KD = 16 * NKS, KS = KD + 4;
  __shared__ __attribute__((aligned(16))) float kl[CT * KS], vt[16 * NVT * CS], bt[4 * KD];
  const int h = blockIdx.x, c = c_first + blockIdx.y;
  const int t0 = c_start[c], n = min(c_start[c + 1] - t0, CT);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4, tok = 16 * wave + r16;
  if (16 * wave >= n) {  // no tokens, nothing that another wave reads
    __syncthreads();
    return;
  }
  const bool there = tok < n;
  const bf16_t* row = p + (int64_t)(t0 + (there ? tok : 0)) * p_stride;
  f32x4_t qh[NKS], kh[NKS];
  Total total[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    const int i = 16 * ks + 4 * kq;
    total[ks] = Total{{1.f, 1.f, 1.f, 1.f}, {0.f, 0.f, 0.f, 0.f}};
    qh[ks] = kh[ks] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (there && i < dk) {
      gate4(row + (H + h) * dk + i, f_bias + h * dk + i, lower + h * dk + i, dk - i, vec != 0, total[ks].hi, kh[ks]);
      const f32x4_t raw = load4(row + h * dk + i, dk - i, vec != 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) qh[ks][j] = Fn<bf16_t>::silu(raw[j]);
    }
  }
  const bool finite = stage_values<NVT>(row + 2 * H * dk + h * dv, there, dv, vec != 0, kq, tok, vt);

  // scores of query r16 against the keys 4 kq + r of the own block
  f32x4_t same = {0.f, 0.f, 0.f, 0.f}, at1 = same, at2 = same, at4 = same, at8 = same;
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    same = mul_add4(kh[ks], qh[ks], same);
    qh[ks] *= total[ks].hi;
    at1 = mul_add4(kh[ks], qh[ks], at1);
    qh[ks] *= widen<1>(r16, total[ks], kh[ks]);
    at2 = mul_add4(kh[ks], qh[ks], at2);
    qh[ks] *= widen<2>(r16, total[ks], kh[ks]);
    at4 = mul_add4(kh[ks], qh[ks], at4);
    qh[ks] *= widen<4>(r16, total[ks], kh[ks]);
    at8 = mul_add4(kh[ks], qh[ks], at8);
    qh[ks] *= widen<8>(r16, total[ks], kh[ks]);
    const int i = 16 * ks + 4 * kq;
    *reinterpret_cast<f32x4_t*>(kl + tok * KS + i) = kh[ks];
    if (r16 == 0) *reinterpret_cast<f32x4_t*>(bt + wave * KD + i) = total[ks].value();
  }
  f32x4_t sc;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = 4 * kq + r, x = r16 ^ s;
    sc[r] = s > r16 ? 0.f : x == 0 ? same[r] : x == 1 ? at1[r] : x < 4 ? at2[r] : x < 8 ? at4[r] : at8[r];
  }
  __syncthreads();

  f32x4_t o[NVT];  // o[m][r] = token r16, column 16 m + 4 kq + r
#pragma unroll
  for (int m = 0; m < NVT; ++m) o[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto values = [&](int b, const f32x4_t& w) {
#pragma unroll
    for (int m = 0; m < NVT; ++m)
      o[m] = mul_add4(*reinterpret_cast<const f32x4_t*>(vt + (16 * m + r16) * CS + 16 * b + 4 * kq), w, o[m]);
  };
  if (__all(finite)) {
    values(wave, sc);
  } else {
    // the own block's later tokens have weight 0, and 0 times an infinity would spoil the earlier ones: finite values as
    // above, the others token by token
    auto usual = [](float v) { return __builtin_fabsf(v) < INFINITY; };
#pragma unroll
    for (int m = 0; m < NVT; ++m) {
      f32x4_t v = *reinterpret_cast<const f32x4_t*>(vt + (16 * m + r16) * CS + 16 * wave + 4 * kq);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = usual(v[j]) ? v[j] : 0.f;
      o[m] = mul_add4(v, sc, o[m]);
    }
#pragma unroll 1
    for (int s = 0; s < 16; ++s) {
      const float mine = (s & 2) ? ((s & 1) ? sc[3] : sc[2]) : ((s & 1) ? sc[1] : sc[0]);
      const float w = __shfl(mine, (s >> 2) * 16 + r16, 64);
#pragma unroll
      for (int m = 0; m < NVT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = vt[(16 * m + 4 * kq + r) * CS + 16 * wave + s];
          if (s <= r16 && !usual(v)) o[m][r] += w * v;
        }
    }
  }
  for (int b = wave - 1; b >= 0; --b) {  // qh: from here on with the decays back to the end of block b
    f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) a = mul_add4(*reinterpret_cast<const f32x4_t*>(kl + (16 * b + r16) * KS + 16 * ks + 4 * kq), qh[ks], a);
    values(b, a);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qh[ks] *= *reinterpret_cast<const f32x4_t*>(bt + b * KD + 16 * ks + 4 * kq);
  }
  const float* S = c_state + ((int64_t)c * H + h) * dv * KD;
#pragma unroll
  for (int m = 0; m < NVT; ++m) {
    const bool ok = 16 * m + r16 < dv;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      f32x4_t a = {0.f, 0.f, 0.f, 0.f};
      if (ok) a = *reinterpret_cast<const f32x4_t*>(S + (16 * m + r16) * KD + 16 * ks + 4 * kq);
      o[m] = mul_add4(a, qh[ks], o[m]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int m = 0; m < NVT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) ss += o[m][r] * o[m][r];
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (!there) return;
  const float inv = Fn<bf16_t>::rsqrt(ss / (float)dv + eps);
  bf16_t* dst = out + ((int64_t)(t0 + tok) * H + h) * dv;
#pragma unroll
  for (int m = 0; m < NVT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = 16 * m + 4 * kq + r;
      if (col < dv) st(dst + col, o[m][r] * inv * ld(norm_w + col));
    }
}

}  // namespace

extern "C" {

// Padded key rows per head (4 KR) for a key size, or 0 when it does not fit (dk > 256).
int sm_gated_delta_rows(int dk) { return dk <= 32 ? 32 : dk <= 64 ? 64 : dk <= 128 ? 128 : dk <= 256 ? 256 : 0; }

// Workspaces (fp32): qn, kn [T, G, KD]; dec [T, H, KD] or [T, H]; beta [T, H]; o_raw [T, H, dv].
// Returns 0, or 1 when the key size does not fit (dk > 256).
int sm_gated_delta_scan(const void* xc, int64_t x_stride, int G, int dk, int H, int dv, const void* beta_raw,
                        int64_t beta_stride, const void* decay_raw, int64_t decay_stride, int per_channel,
                        const float* A, const float* dt_bias, const void* gate_raw, int64_t gate_stride,
                        int gate_sigmoid, const void* norm_w, float eps, float* state, const int* seq_start,
                        const int* seq_slot, const int* seq_init, void* out, float* qn, float* kn, float* dec,
                        float* beta, float* o_raw, int T, int nseq, int f32, hipStream_t stream) {
  if (nseq == 0 || T == 0) return 0;
  const int KD = sm_gated_delta_rows(dk);
  if (KD == 0) return 1;
  const int voff = 2 * G * dk;
  // 16 columns x 4 row groups per wave when the step brings many waves anyway (decode: 64-byte pieces of
  // the state's rows); 8 x 8 when it brings few (a prompt): twice the waves, half the work of each
  const bool wide = (int64_t)nseq * H * ((dv + 15) / 16) >= 1024;
  const int cpw = wide ? 16 : 8;
  const dim3 grid(H * ((dv + cpw - 1) / cpw), nseq);
  const dim3 ogrid(T, std::max(1, std::min((H + 3) / 4, 4096 / T)));
#define SM_GO(TYPE, KR, RG, CH)                                                                                     \
  hipLaunchKernelGGL((gated_delta_scan_kernel<TYPE, KR, RG, CH, (KR * RG <= 128 ? 16 : 8)>), grid, dim3(64), 0, stream, \
                     qn, kn, dec, beta, (const TYPE*)xc, x_stride, voff, G, dk, H, dv, state, seq_start, seq_slot,  \
                     seq_init, o_raw)
#define SM_RG(TYPE, KD_, CH)              \
  if (wide) SM_GO(TYPE, KD_ / 4, 4, CH);  \
  else SM_GO(TYPE, KD_ / 8, 8, CH)
#define SM_KR(TYPE, CH)                           \
  if (KD == 32) { SM_RG(TYPE, 32, CH); }          \
  else if (KD == 64) { SM_RG(TYPE, 64, CH); }     \
  else if (KD == 128) { SM_RG(TYPE, 128, CH); }   \
  else { SM_RG(TYPE, 256, CH); }
#define SM_ALL(TYPE)                                                                                                \
  hipLaunchKernelGGL((delta_prep_kernel<TYPE>), dim3(T), dim3(NT), 0, stream, (const TYPE*)xc, x_stride, G, dk, KD, \
                     H, (const TYPE*)beta_raw, beta_stride, (const TYPE*)decay_raw, decay_stride, per_channel, A,   \
                     dt_bias, qn, kn, dec, beta);                                                                   \
  if (per_channel) { SM_KR(TYPE, true) }                                                                           \
  else { SM_KR(TYPE, false) }                                                                                      \
  hipLaunchKernelGGL((delta_out_kernel<TYPE>), ogrid, dim3(NT), 0, stream, o_raw, (const TYPE*)gate_raw,            \
                     gate_stride, gate_sigmoid, (const TYPE*)norm_w, eps, H, dv, (TYPE*)out)
  if (f32) { SM_ALL(float); }
  else { SM_ALL(bf16_t); }
#undef SM_ALL
#undef SM_KR
#undef SM_RG
#undef SM_GO
  return 0;
}

// Key rows per head of the prompt form's scratch, or 0 where the sizes are outside its compiled forms (float32,
// dk or dv > 128).
int sm_hgrn2_chunk_rows(int dk, int dv, int f32) {
  return f32 || dv > 128 ? 0 : dk <= 32 ? 32 : dk <= 64 ? 64 : dk <= 128 ? 128 : 0;
}

// HGRN2 over the projection p = [q | f | v] (H dk, H dk, H dv columns). Workspaces (fp32): qn, kn, dec
// [T, H, KD]; o_raw [T, H, dv]. Returns 0, or 1 when the key size does not fit (dk > 256).
// nc > 0: the chunked form. c_start [nc + 1] bounds the chunks (every run cut into pieces), c_slot = 0 .. nc - 1,
// c_zero / c_one [nc] are all 0 / all 1, s_chunk0 [nseq + 1] bounds each sequence's chunks; c_state
// [nc, H, dk, dv] and c_decay [nc, H, KD] are fp32 scratch. Where sm_hgrn2_chunk_rows gives the rows of the matrix-core form,
// they have [nc, H, dv, rows] and [nc, H, rows]; the first nd sequences, of one token each, go token by token there (a chunk
// costs about as much for one token as for 64), and qn, kn, dec and o_raw hold their nd tokens alone.
int sm_hgrn2_scan(const void* p, int64_t p_stride, int H, int dk, int dv, const float* f_bias, const float* lower,
                  const void* norm_w, float eps, float* state, const int* seq_start, const int* seq_slot,
                  const int* seq_init, void* out, float* qn, float* kn, float* dec, float* o_raw, int T, int nseq,
                  int f32, int nd, int nc, const int* c_start, const int* c_slot, const int* c_zero, const int* c_one,
                  const int* s_chunk0, float* c_state, float* c_decay, hipStream_t stream) {
  if (nseq == 0 || T == 0) return 0;
  const int rows = nc > nd ? sm_hgrn2_chunk_rows(dk, dv, f32) : 0;
  if (rows > 0) {
    if (nd > 0)
      sm_hgrn2_scan(p, p_stride, H, dk, dv, f_bias, lower, norm_w, eps, state, seq_start, seq_slot, seq_init, out, qn, kn, dec,
                    o_raw, nd, nd, f32, 0, 0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, stream);
    const int vec = dk % 4 == 0 && dv % 4 == 0 && p_stride % 4 == 0 && ((uintptr_t)p & 7) == 0 &&
                    (((uintptr_t)f_bias | (uintptr_t)lower) & 15) == 0;
    const dim3 cgrid(H, nc - nd), lgrid((unsigned)(((int64_t)H * dv * rows + NT - 1) / NT), nseq - nd);
#define SM_GO(NKS, NVT)                                                                                               \
  do {                                                                                                                \
    hipLaunchKernelGGL((hgrn2_chunk_kernel<NKS, NVT>), cgrid, dim3(NT), 0, stream, (const bf16_t*)p, p_stride, H, dk, \
                       dv, vec, f_bias, lower, c_start, nd, c_state, c_decay);                                        \
    hipLaunchKernelGGL(hgrn2_link_kernel, lgrid, dim3(NT), 0, stream, c_state, c_decay, s_chunk0, nd, H, dk, dv,      \
                       rows, state, seq_slot, seq_init);                                                              \
    hipLaunchKernelGGL((hgrn2_read_kernel<NKS, NVT>), cgrid, dim3(NT), 0, stream, (const bf16_t*)p, p_stride, H, dk,  \
                       dv, vec, f_bias, lower, c_start, nd, c_state, (const bf16_t*)norm_w, eps, (bf16_t*)out);       \
  } while (0)
    if (rows == 32 && dv <= 64) SM_GO(2, 4);
    else if (rows == 32) SM_GO(2, 8);
    else if (rows == 64 && dv <= 64) SM_GO(4, 4);
    else if (rows == 64) SM_GO(4, 8);
    else if (dv <= 64) SM_GO(8, 4);
    else SM_GO(8, 8);
#undef SM_GO
    return 0;
  }
  const int KD = sm_gated_delta_rows(dk);
  if (KD == 0) return 1;
  const int voff = 2 * H * dk;
  const int nrun = nc > 0 ? nc : nseq;  // runs the scan kernel sees
  const bool wide = (int64_t)nrun * H * ((dv + 15) / 16) >= 1024;
  const int cpw = wide ? 16 : 8;
  const dim3 grid(H * ((dv + cpw - 1) / cpw), nrun);
  const dim3 pgrid(T, std::max(1, std::min((H * KD + NT - 1) / NT, 4096 / T)));
  const dim3 ogrid(T, std::max(1, std::min((H + 3) / 4, 4096 / T)));
#define SM_GO(TYPE, KR, RG, OUT_, ST, START, SLOT, INIT)                                                              \
  hipLaunchKernelGGL((gated_delta_scan_kernel<TYPE, KR, RG, true, (KR * RG <= 128 ? 16 : 8), false, OUT_>), grid,      \
                     dim3(64), 0, stream, qn, kn, dec, nullptr, (const TYPE*)p, p_stride, voff, H, dk, H, dv, ST,      \
                     START, SLOT, INIT, o_raw, c_decay)
#define SM_RG(TYPE, KD_, ...)                      \
  if (wide) SM_GO(TYPE, KD_ / 4, 4, __VA_ARGS__);  \
  else SM_GO(TYPE, KD_ / 8, 8, __VA_ARGS__)
#define SM_KD(TYPE, ...)                                     \
  if (KD == 32) { SM_RG(TYPE, 32, __VA_ARGS__); }            \
  else if (KD == 64) { SM_RG(TYPE, 64, __VA_ARGS__); }       \
  else if (KD == 128) { SM_RG(TYPE, 128, __VA_ARGS__); }     \
  else { SM_RG(TYPE, 256, __VA_ARGS__); }
#define SM_ALL(TYPE)                                                                                                 \
  hipLaunchKernelGGL((hgrn2_prep_kernel<TYPE>), pgrid, dim3(NT), 0, stream, (const TYPE*)p, p_stride, H, dk, KD,      \
                     f_bias, lower, qn, kn, dec);                                                                    \
  if (nc > 0) {                                                                                                      \
    SM_KD(TYPE, false, c_state, c_start, c_slot, c_zero)                                                             \
    hipLaunchKernelGGL(chunk_link_kernel, dim3((unsigned)std::min<int64_t>(((int64_t)H * dk * dv + NT - 1) / NT, 2048), \
                                               nseq), dim3(NT), 0, stream, c_state, c_decay, s_chunk0, H, dk, dv, KD, \
                       state, seq_slot, seq_init);                                                                   \
    SM_KD(TYPE, true, c_state, c_start, c_slot, c_one)                                                               \
  } else {                                                                                                           \
    SM_KD(TYPE, true, state, seq_start, seq_slot, seq_init)                                                          \
  }                                                                                                                  \
  hipLaunchKernelGGL((delta_out_kernel<TYPE>), ogrid, dim3(NT), 0, stream, o_raw, (const TYPE*)nullptr, (int64_t)0, 0, \
                     (const TYPE*)norm_w, eps, H, dv, (TYPE*)out)
  if (f32) { SM_ALL(float); }
  else { SM_ALL(bf16_t); }
#undef SM_ALL
#undef SM_KD
#undef SM_RG
#undef SM_GO
  return 0;
}

}  // extern "C"
