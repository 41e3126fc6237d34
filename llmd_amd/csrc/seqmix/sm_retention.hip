// Retention: linear attention whose state S [dk, dv] per head (fp32) forgets with a fixed decay. Over a step's
// per-sequence token runs, each continuing the state in its slot (seq_slot) or starting from zero (seq_init == 0):
//
//   q, k rotated on their first rot_dims dimensions (pairs (i, i + rot_dims / 2)), k times dk^-1/2
//   S <- decay S + k v^T;  o = S^T q;  out = o / rms(o) * silu(g)
//
// from the fused projection rows [q | k | v (| g)]; everything between the projections and ``out`` is fp32.
//
// retention_step  : sequences that bring one token. One workgroup per (head, sequence) rotates q and k, streams S
//                   once (16-byte pieces, a thread keeps its columns), and norms and gates the read-out.
// Longer runs are cut into chunks of at most C = 64 tokens. A chunk of n tokens that starts from S gives
//   o_i = decay^(i+1) S^T q_i + sum_{j <= i} decay^(i-j) (q_i . k_j) v_j,   S' = decay^n S + sum_j decay^(n-1-j) k_j v_j^T
// so all products are matrix products. They run on v_mfma_f32_16x16x4_f32: operands and sums are fp32. bf16 rows of the usual head sizes
// take the kernels *_parts further down instead.
// retention_chunk : every chunk's own part of its final state, L = sum_j decay^(n-1-j) k_j v_j^T.
// retention_link  : walks a sequence's chunks in order, S_(c+1) = decay^n S_c + L_c; leaves every chunk's start
//                   state where its L was and the run's final state in the slot.
// retention_out   : a chunk's read-outs; workgroup = 64 queries (16 per wave) x up to 256 columns. The weights of the
//                   second product stay in the registers the scores arrive in. Norm and gate are fused when one
//                   workgroup holds all of a head's columns, else retention_norm follows.
// In all of them the contraction index is dealt so that an operand's four consecutive elements belong to one lane:
// step e of a group of 16 takes element 4 kq + e from lane group kq, on both sides.
#include "moe_tile.h"
#include "seqmix_common.h"
#include <algorithm>

using namespace sm;

namespace {

constexpr int NT = 256;
constexpr int C = 64;         // tokens per chunk
constexpr int DB = 64;        // key dimensions staged at a time
constexpr int QS = DB + 4;    // LDS row stride of the keys
constexpr int MAXCOLS = 256;  // value columns of a workgroup

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void ld4(const float* p, float (&v)[4]) {
  const float4 t = *reinterpret_cast<const float4*>(p);
  v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void ld4(const bf16_t* p, float (&v)[4]) {
  const uint2 t = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(t.x << 16); v[1] = __uint_as_float(t.x & 0xffff0000u);
  v[2] = __uint_as_float(t.y << 16); v[3] = __uint_as_float(t.y & 0xffff0000u);
}

struct Rot {
  const int64_t* positions;
  const float* cos_sin;  // [max_pos, dims] = [cos | sin]
  int dims;              // 0: no rotation
};

// Element e of a head's rotated row.
template <typename T>
__device__ __forceinline__ float rot1(const T* row, int e, const float* cs, int half) {
  const float x = ld(row + e);
  if (e >= 2 * half) return x;
  const bool first = e < half;
  const float xp = ld(row + (first ? e + half : e - half));
  const int f = first ? e : e - half;
  const float c = cs[f], s = cs[half + f];
  return first ? x * c - xp * s : x * c + xp * s;
}

// Elements e .. e + 3, zero past dk. VEC (dk and half multiples of four, rows aligned for it): all loads are
// unconditional, from clamped places, so that those of several calls are in flight together.
template <typename T, bool VEC>
__device__ __forceinline__ void rot4(const T* row, int e, int dk, const float* cs, int half, float (&v)[4]) {
  if constexpr (!VEC) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = e + i < dk ? rot1(row, e + i, cs, half) : 0.f;
  } else {
    const int ec = min(e, dk - 4);
    ld4(row + ec, v);
    if (half > 0) {
      const bool first = ec < half, in = ec < 2 * half;
      const int f = in ? (first ? ec : ec - half) : 0;
      float p[4], c[4], s[4];
      ld4(row + (in ? (first ? ec + half : ec - half) : ec), p);
      ld4(cs + f, c);
      ld4(cs + half + f, s);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = in ? (first ? v[i] * c[i] - p[i] * s[i] : v[i] * c[i] + p[i] * s[i]) : v[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = e < dk ? v[i] : 0.f;
  }
}

// ---------------------------------------------------------------------------------------------
// VEC columns per thread; ncg = column groups side by side, RG = row groups (threads past RG * ncg idle).
template <typename T, int VEC>
__global__ __launch_bounds__(NT) void retention_step_kernel(const T* __restrict__ p, int64_t stride, int H, int dk,
                                                            int dv, int gate, Rot rot, const float* __restrict__ powers,
                                                            int pw_stride, float eps, float* __restrict__ state,
                                                            const int* __restrict__ seq_start,
                                                            const int* __restrict__ seq_slot,
                                                            const int* __restrict__ seq_init, T* __restrict__ out,
                                                            int ncg, int RG) {
  extern __shared__ float lds[];
  __shared__ float red[NT / 64];
  const int h = blockIdx.x, s = blockIdx.y;
  const int64_t t = seq_start[s];
  const bool init = seq_init[s] != 0;
  float* sp = state + ((int64_t)seq_slot[s] * H + h) * dk * dv;
  float *sq = lds, *sk = lds + dk, *so = lds + 2 * dk;  // so [RG, dv]
  const T* row = p + t * stride;
  const int rg = threadIdx.x / ncg, cg = threadIdx.x - rg * ncg;
  constexpr int U = 8;  // rows of the state in flight
  float S[U][VEC];
  auto load = [&](int r0, int col) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = r0 + u * RG;
#pragma unroll
      for (int i = 0; i < VEC; ++i) S[u][i] = 0.f;
      if (init && r < dk) {
        if constexpr (VEC == 4) ld4(sp + (int64_t)r * dv + col, S[u]);
        else S[u][0] = sp[(int64_t)r * dv + col];
      }
    }
  };
  if (rg < RG) load(rg, cg * VEC);  // the first piece is on its way while the keys and queries are rotated
  const int half = rot.dims >> 1;
  const float* cs = rot.dims ? rot.cos_sin + rot.positions[t] * rot.dims : nullptr;
  const float kscale = 1.f / sqrtf((float)dk);
  const float decay = powers[h * pw_stride + 1];
  for (int e = threadIdx.x; e < 2 * dk; e += NT) {
    const bool is_q = e < dk;
    const int d = is_q ? e : e - dk;
    const float x = rot1(row + (is_q ? h : H + h) * dk, d, cs, half);
    lds[e] = is_q ? x : x * kscale;
  }
  __syncthreads();
  const T* vrow = row + 2 * H * dk + h * dv;
  if (rg < RG) {
    for (int col = cg * VEC; col < dv; col += ncg * VEC) {
      if (col != cg * VEC) load(rg, col);
      float v[VEC], o[VEC];
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        v[i] = ld(vrow + col + i);
        o[i] = 0.f;
      }
      for (int r0 = rg; r0 < dk; r0 += RG * U) {
        if (r0 != rg) load(r0, col);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int r = r0 + u * RG;
          if (r >= dk) continue;
          const float k = sk[r], q = sq[r];
#pragma unroll
          for (int i = 0; i < VEC; ++i) {
            S[u][i] = decay * S[u][i] + k * v[i];
            o[i] += S[u][i] * q;
          }
          if constexpr (VEC == 4)
            *reinterpret_cast<float4*>(sp + (int64_t)r * dv + col) = make_float4(S[u][0], S[u][1], S[u][2], S[u][3]);
          else
            sp[(int64_t)r * dv + col] = S[u][0];
        }
      }
#pragma unroll
      for (int i = 0; i < VEC; ++i) so[rg * dv + col + i] = o[i];
    }
  }
  __syncthreads();
  const T* grow = row + 2 * H * dk + H * dv + h * dv;
  const float g0 = gate && (int)threadIdx.x < dv ? ld(grow + threadIdx.x) : 0.f;
  float ss = 0.f;
  for (int e = threadIdx.x; e < dv; e += NT) {  // a thread reads back only what it sums here
    float a = 0.f;
    for (int g = 0; g < RG; ++g) a += so[g * dv + e];
    so[e] = a;
    ss += a * a;
  }
  const float inv = 1.f / sqrtf(block_sum<NT>(ss, red) / (float)dv + eps);
  for (int e = threadIdx.x; e < dv; e += NT) {
    float o = so[e] * inv;
    if (gate) o *= Fn<T>::silu(e < NT ? g0 : ld(grow + e));
    st(out + (t * H + h) * dv + e, o);
  }
}

// ---------------------------------------------------------------------------------------------
// Stage CB value columns [col0, col0 + CB) of ROWS tokens t0 .. (rows past n and columns past dv are zero).
template <typename T, int CB, int ROWS, bool VEC>
__device__ __forceinline__ void stage_v(const T* __restrict__ p, int64_t stride, int64_t t0, int n, int voff, int col0,
                                        int dv, float* sV) {
  constexpr int BS = CB + 4;
#pragma unroll
  for (int e0 = 0; e0 < ROWS * (CB / 4); e0 += NT) {
    const int e = e0 + threadIdx.x;
    const int j = e / (CB / 4), c = (e - j * (CB / 4)) * 4;
    const T* src = p + (t0 + min(j, n - 1)) * stride + voff;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      ld4(src + min(col0 + c, dv - 4), v);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = j < n && col0 + c < dv ? v[i] : 0.f;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j < n && col0 + c + i < dv) v[i] = ld(src + col0 + c + i);
    }
    *reinterpret_cast<float4*>(&sV[j * BS + c]) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// L = sum_j decay^(n-1-j) k_j v_j^T of chunk c0 + blockIdx.x, head blockIdx.y; blockIdx.z: block of DB key rows x CB columns.
template <typename T, int NCB, bool VEC>
__global__ __launch_bounds__(NT) void retention_chunk_kernel(const T* __restrict__ p, int64_t stride, int H, int dk,
                                                             int dv, Rot rot, const float* __restrict__ powers,
                                                             int pw_stride, const int* __restrict__ c_start, int c0,
                                                             float* __restrict__ c_state) {
  constexpr int CB = 16 * NCB, BS = CB + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *sK = lds, *sV = lds + C * QS;
  const int c = blockIdx.x, h = blockIdx.y;
  const int ncb = (dv + CB - 1) / CB;
  const int d0 = (int)(blockIdx.z / ncb) * DB, col0 = (int)(blockIdx.z % ncb) * CB;
  const int64_t t0 = c_start[c0 + c];
  const int n = c_start[c0 + c + 1] - (int)t0;
  const int half = rot.dims >> 1;
  const float kscale = 1.f / sqrtf((float)dk);
  const float* pw = powers + (int64_t)h * pw_stride;
  const int64_t pos0 = rot.positions[t0];  // a chunk's positions follow each other
#pragma unroll
  for (int e0 = 0; e0 < C * (DB / 4); e0 += NT) {
    const int e = e0 + threadIdx.x;
    const int j = e / (DB / 4), d = (e - j * (DB / 4)) * 4, jc = min(j, n - 1);
    float v[4];
    rot4<T, VEC>(p + (t0 + jc) * stride + (H + h) * dk, d0 + d, dk, rot.cos_sin + (pos0 + jc) * rot.dims, half, v);
    const float w = j < n ? kscale * pw[n - 1 - jc] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = j < n ? v[i] * w : 0.f;
    *reinterpret_cast<float4*>(&sK[j * QS + d]) = make_float4(v[0], v[1], v[2], v[3]);
  }
  stage_v<T, CB, C, VEC>(p, stride, t0, n, 2 * H * dk + h * dv, col0, dv, sV);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  if (d0 + wave * 16 >= dk) return;
  f32x4_t acc[NCB];
#pragma unroll
  for (int m = 0; m < NCB; ++m) acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < n; j0 += 16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + 4 * kq + e;
      const float a = sK[j * QS + wave * 16 + r16];
#pragma unroll
      for (int m = 0; m < NCB; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, sV[j * BS + m * 16 + r16], acc[m], 0, 0, 0);
    }
  }
  float* dst = c_state + ((int64_t)c * H + h) * dk * dv;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int d = d0 + wave * 16 + kq * 4 + r;
    if (d >= dk) continue;
#pragma unroll
    for (int m = 0; m < NCB; ++m) {
      const int col = col0 + m * 16 + r16;
      if (col < dv) dst[(int64_t)d * dv + col] = acc[m][r];
    }
  }
}

// Sequence s0 + blockIdx.y: its chunks in order, VEC elements of the state per thread.
template <int VEC>
__global__ __launch_bounds__(NT) void retention_link_kernel(float* __restrict__ c_state, const int* __restrict__ c_start,
                                                            const int* __restrict__ s_chunk0, int c0, int s0, int H,
                                                            int64_t per_head, const float* __restrict__ powers,
                                                            int pw_stride, float* __restrict__ state,
                                                            const int* __restrict__ seq_slot,
                                                            const int* __restrict__ seq_init) {
  const int s = s0 + blockIdx.y;
  const int64_t total = per_head * H;
  const int64_t e = ((int64_t)blockIdx.x * NT + threadIdx.x) * VEC;
  if (e >= total) return;
  const float* pw = powers + (e / per_head) * pw_stride;  // VEC divides a head's elements
  const int lo = s_chunk0[s], hi = s_chunk0[s + 1];
  if (lo >= hi) return;
  float* sp = state + (int64_t)seq_slot[s] * total + e;
  float S[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) S[i] = 0.f;
  if (seq_init[s]) {
    if constexpr (VEC == 4) ld4(sp, S);
    else S[0] = sp[0];
  }
  constexpr int U = 16;  // chunks in flight
  const float d_full = pw[C], d_last = pw[c_start[hi] - c_start[hi - 1]];  // all chunks but a run's last are whole
  for (int cb = lo; cb < hi; cb += U) {
    float L[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float* src = c_state + (int64_t)(min(cb + u, hi - 1) - c0) * total + e;
      if constexpr (VEC == 4) ld4(src, L[u]);
      else L[u][0] = src[0];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (cb + u < hi) {
        float* dst = c_state + (int64_t)(cb + u - c0) * total + e;
        if constexpr (VEC == 4) *reinterpret_cast<float4*>(dst) = make_float4(S[0], S[1], S[2], S[3]);
        else dst[0] = S[0];
        const float d = cb + u == hi - 1 ? d_last : d_full;
#pragma unroll
        for (int i = 0; i < VEC; ++i) S[i] = d * S[i] + L[u][i];
      }
  }
  if constexpr (VEC == 4) *reinterpret_cast<float4*>(sp) = make_float4(S[0], S[1], S[2], S[3]);
  else sp[0] = S[0];
}

// The read-outs of chunk c0 + blockIdx.x, head blockIdx.y, columns CB blockIdx.z ..; c_state holds the chunks' start states.
// A wave's 16 rotated queries go from global memory to its registers; keys (OB dimensions at a time), the state's
// rows (OB at a time) and the values (OB tokens at a time) pass through LDS in small pieces, so that several
// workgroups share a CU and hide each other's loads.
constexpr int OB = 32, OS = OB + 4;

template <typename T, int NCB, bool VEC>
__global__ __launch_bounds__(NT, NCB <= 4 ? 4 : NCB <= 8 ? 3 : 2) void retention_out_kernel(const T* __restrict__ p, int64_t stride, int H, int dk,
                                                           int dv, int gate, Rot rot, const float* __restrict__ powers,
                                                           int pw_stride, float eps, const int* __restrict__ c_start,
                                                           int c0, const float* __restrict__ c_state,
                                                           T* __restrict__ out, float* __restrict__ o_raw) {
  constexpr int CB = 16 * NCB, BS = CB + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float sP[C + 1];
  float *sK = lds, *sB = lds + C * OS;  // sK [64 keys, OB]; sB [OB, CB]: a piece of the state, then of the values
  const int c = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * CB;
  const int64_t t0 = c_start[c0 + c];
  const int n = c_start[c0 + c + 1] - (int)t0;
  const int half = rot.dims >> 1;
  const float kscale = 1.f / sqrtf((float)dk);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, kq = lane >> 4;
  if (threadIdx.x <= C) sP[threadIdx.x] = powers[(int64_t)h * pw_stride + threadIdx.x];
  const float* S0 = c_state + ((int64_t)c * H + h) * dk * dv;
  const int64_t pos0 = rot.positions[t0];  // a chunk's positions follow each other
  const int qi = wave * 16 + r16, qc = min(qi, n - 1);
  const T* q_row = p + (t0 + qc) * stride + h * dk;
  const float* q_cs = rot.cos_sin + (pos0 + qc) * rot.dims;
  f32x4_t o[NCB], w[4];  // o: rows 16 wave + 4 kq + r, column 16 m + r16; w[jb]: key 16 jb + 4 kq + r of query 16 wave + r16
#pragma unroll
  for (int m = 0; m < NCB; ++m) o[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) w[jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int d0 = 0; d0 < dk; d0 += OB) {
    float a[OB / 16][4];  // this lane's query, dimensions d0 + 16 i + 4 kq .. (a row past n repeats the last one)
#pragma unroll
    for (int i = 0; i < OB / 16; ++i) rot4<T, VEC>(q_row, d0 + 16 * i + 4 * kq, dk, q_cs, half, a[i]);
    if (d0 > 0) __syncthreads();  // the previous piece is read
#pragma unroll
    for (int e0 = 0; e0 < C * (OB / 4); e0 += NT) {
      const int e = e0 + threadIdx.x;
      const int j = e / (OB / 4), d = (e - j * (OB / 4)) * 4, jc = min(j, n - 1);
      float b[4];
      rot4<T, VEC>(p + (t0 + jc) * stride + (H + h) * dk, d0 + d, dk, rot.cos_sin + (pos0 + jc) * rot.dims, half, b);
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = j < n ? b[i] * kscale : 0.f;
      *reinterpret_cast<float4*>(&sK[j * OS + d]) = make_float4(b[0], b[1], b[2], b[3]);
    }
#pragma unroll
    for (int e0 = 0; e0 < OB * (CB / 4); e0 += NT) {
      const int e = e0 + threadIdx.x;
      const int d = e / (CB / 4), cc = (e - d * (CB / 4)) * 4;
      const float* src = S0 + (int64_t)min(d0 + d, dk - 1) * dv;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if constexpr (VEC) {
        ld4(src + min(col0 + cc, dv - 4), v);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = d0 + d < dk && col0 + cc < dv ? v[i] : 0.f;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (d0 + d < dk && col0 + cc + i < dv) v[i] = src[col0 + cc + i];
      }
      *reinterpret_cast<float4*>(&sB[d * BS + cc]) = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OB / 16; ++i) {
      if (d0 + 16 * i >= dk) break;
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        if (jb > wave) break;  // keys after every query of this wave
        float b[4];
        ld4(&sK[(jb * 16 + r16) * OS + 16 * i + 4 * kq], b);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[e], a[i][e], w[jb], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < NCB; ++m)
          o[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], sB[(16 * i + 4 * kq + e) * BS + m * 16 + r16], o[m], 0, 0, 0);
    }
  }
  // decay of the state's part by the row, of a weight by the distance
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float d = sP[wave * 16 + kq * 4 + r + 1];
#pragma unroll
    for (int m = 0; m < NCB; ++m) o[m][r] *= d;
  }
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int dist = wave * 16 + r16 - (jb * 16 + kq * 4 + r);
      w[jb][r] = dist >= 0 ? w[jb][r] * sP[max(dist, 0)] : 0.f;
    }
#pragma unroll
  for (int j0 = 0; j0 < C; j0 += OB) {
    if (j0 >= n) break;
    __syncthreads();  // the previous piece is read
    stage_v<T, CB, OB, VEC>(p, stride, t0 + j0, n - j0, 2 * H * dk + h * dv, col0, dv, sB);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < OB / 16; ++i) {
      const int jb = j0 / 16 + i;
      if (jb > wave) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < NCB; ++m)
          o[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[jb][e], sB[(16 * i + 4 * kq + e) * BS + m * 16 + r16], o[m], 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = wave * 16 + kq * 4 + r;
    const int64_t t = t0 + i;
    if (o_raw != nullptr) {
      if (i < n) {
#pragma unroll
        for (int m = 0; m < NCB; ++m) {
          const int col = col0 + m * 16 + r16;
          if (col < dv) o_raw[(t * H + h) * dv + col] = o[m][r];
        }
      }
      continue;
    }
    float ss = 0.f;  // columns past dv are zero
#pragma unroll
    for (int m = 0; m < NCB; ++m) ss += o[m][r] * o[m][r];
#pragma unroll
    for (int x = 8; x > 0; x >>= 1) ss += __shfl_xor(ss, x, 64);
    const float inv = 1.f / sqrtf(ss / (float)dv + eps);
    float g[NCB];  // the row's gates: loads from clamped places, all in flight together
    if (gate) {
      const T* grow = p + (t0 + min(i, n - 1)) * stride + 2 * H * dk + H * dv + h * dv;
#pragma unroll
      for (int m = 0; m < NCB; ++m) g[m] = ld(grow + min(m * 16 + r16, dv - 1));
#pragma unroll
      for (int m = 0; m < NCB; ++m) o[m][r] *= Fn<T>::silu(g[m]);
    }
    if (i >= n) continue;
#pragma unroll
    for (int m = 0; m < NCB; ++m) {
      const int col = m * 16 + r16;
      if (col < dv) st(out + (t * H + h) * dv + col, o[m][r] * inv);
    }
  }
}

// out = o / rms(o) * silu(g) for tokens t0 + blockIdx.x; a wave per head.
template <typename T>
__global__ __launch_bounds__(NT) void retention_norm_kernel(const float* __restrict__ o_raw, const T* __restrict__ p,
                                                            int64_t stride, int H, int dk, int dv, int gate, float eps,
                                                            const int* __restrict__ first, T* __restrict__ out) {
  const int64_t t = *first + (int64_t)blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int h = blockIdx.y * (NT / 64) + wave; h < H; h += gridDim.y * (NT / 64)) {
    const float* orow = o_raw + (t * H + h) * dv;
    float ss = 0.f;
    for (int e = lane; e < dv; e += 64) ss += orow[e] * orow[e];
    const float inv = 1.f / sqrtf(wave_sum(ss) / (float)dv + eps);
    for (int e = lane; e < dv; e += 64) {
      float v = orow[e] * inv;
      if (gate) v *= Fn<T>::silu(ld(p + t * stride + 2 * H * dk + H * dv + h * dv + e));
      st(out + (t * H + h) * dv + e, v);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same two products on v_mfma_f32_16x16x32_bf16, for bf16 rows: numbers that are fp32 (rotated q and k, weights, the state) as
// three bf16 parts, times 2^24 (moe_tile.h says why); v is bf16 as it is, so its products take three instructions and are exact, those of
// two fp32 numbers six. Sums that are not finite (infinities, NaN, numbers that overflow so scaled) are done again
// number by number. The contraction index is dealt to the lane groups in eights; a lane's eight are one 16-byte piece in LDS.
// Bound by the chunks' states (a head's 128 KB written twice and read twice per 64 tokens: here, by retention_link in between and by
// retention_out) and by the chain of loads and barriers of a
// workgroup; the fp32 instructions alone had taken half of the time, loads one after the other most of the rest.
// us, chunk + out, 16 heads of 128 x 256: 901 + 844 + 787 tokens 65 + 100 -> 38 + 53 over and over, 42 + 58 in a step behind its other
// kernels. States off 64 bits: less than before (exact
// products, a sixteenth of the roundings).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
constexpr float UP1 = 0x1p-24f;  // of sums with one factor times 2^24
struct Parts {
  u32x4_t p[3];  // 8 elements: largest part first
};
// (As vectors of two: hipcc rounds scalar casts twice, and what asm writes it hands to the matrix units too early.)
__device__ __forceinline__ Parts split_vals(const float (&a)[4], const float (&b)[4]) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  f32x2_t x[4] = {{a[0], a[1]}, {a[2], a[3]}, {b[0], b[1]}, {b[2], b[3]}};
  Parts r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x[j] *= moe_tile::SPLIT_UP;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(x[j], bf16x2_t));
      x[j][0] -= __uint_as_float(w << 16), x[j][1] -= __uint_as_float(w & 0xffff0000u);
      r.p[i][j] = w;
    }
  }
  return r;
}

__device__ __forceinline__ f32x4_t mfma_bf(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma_six(const u32x4_t (&a)[3], const u32x4_t (&b)[3], f32x4_t c) {
  c = mfma_bf(a[2], b[0], c);
  c = mfma_bf(a[0], b[2], c);
  c = mfma_bf(a[1], b[1], c);
  c = mfma_bf(a[1], b[0], c);
  c = mfma_bf(a[0], b[1], c);
  return mfma_bf(a[0], b[0], c);
}
// Eight rows of W columns (rows[i]: the columns' first bits) to W pieces of eight rows each
__device__ __forceinline__ uint32_t pick(uint32_t a, uint32_t b, bool high) {
  return high ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
}
template <int W>
__device__ __forceinline__ u32x4_t column(const uint32_t (&rows)[8][W / 2], int i) {
  u32x4_t r;
#pragma unroll
  for (int x = 0; x < 4; ++x) r[x] = pick(rows[2 * x][i / 2], rows[2 * x + 1][i / 2], i & 1);
  return r;
}
// Places of column c's piece where a lane writes W consecutive columns: eight lanes' pieces in banks of their own
template <int W>
__device__ __forceinline__ int place(int c) {
  return W == 4 ? (c & ~3) | ((c + (c >> 3)) & 3) : c ^ ((c >> 3) & 1);
}
// W columns of eight tokens, token(i) the place of the i-th one in the chunk; zeros past n. rv: the chunk's values, col: the first column.
// SHARED: a wave's tokens are the same, their places go beside the address that all lanes share (as pointers hipcc keeps all eight in
// registers and spills).
template <int W, bool SHARED, typename F>
__device__ __forceinline__ void load_v(__amdgpu_buffer_rsrc_t rv, int64_t stride, int col, int n, F token, uint32_t (&rows)[8][W / 2]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = token(i), at = min(j, n - 1) * (int)stride * 2;
    if constexpr (W == 4) {
      const auto t = __builtin_amdgcn_raw_buffer_load_b64(rv, col * 2 + (SHARED ? 0 : at), SHARED ? at : 0, 0);
      rows[i][0] = t[0], rows[i][1] = t[1];
    } else {
      rows[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rv, col * 2 + (SHARED ? 0 : at), SHARED ? at : 0, 0);
    }
#pragma unroll
    for (int x = 0; x < W / 2; ++x) rows[i][x] = j < n ? rows[i][x] : 0;
  }
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000);
}

// Four elements of a row and what their rotation takes. Loads come first and from clamped places, so that those of many calls are in
// flight together; without a rotation (dims 0) cos_sin points at any sixteen bytes.
struct Raw4 {
  uint2 x, p;
  float4 c, s;
};
__device__ __forceinline__ Raw4 load_raw(const bf16_t* row, int e, int dk, const float* cs, int half) {
  const int ec = min(e, dk - 4), f = ec < half ? ec : ec < 2 * half ? ec - half : 0;
  Raw4 r;
  r.x = *reinterpret_cast<const uint2*>(row + ec);
  r.p = *reinterpret_cast<const uint2*>(row + (ec < half ? ec + half : ec < 2 * half ? ec - half : ec));
  r.c = *reinterpret_cast<const float4*>(cs + f);
  r.s = *reinterpret_cast<const float4*>(cs + half + f);
  return r;
}
__device__ __forceinline__ void rotate(const Raw4& r, int e, int dk, int half, float (&v)[4]) {
  const float x[4] = {__uint_as_float(r.x.x << 16), __uint_as_float(r.x.x & 0xffff0000u), __uint_as_float(r.x.y << 16), __uint_as_float(r.x.y & 0xffff0000u)};
  const float p[4] = {__uint_as_float(r.p.x << 16), __uint_as_float(r.p.x & 0xffff0000u), __uint_as_float(r.p.y << 16), __uint_as_float(r.p.y & 0xffff0000u)};
  const float c[4] = {r.c.x, r.c.y, r.c.z, r.c.w}, s[4] = {r.s.x, r.s.y, r.s.z, r.s.w};
  const int ec = min(e, dk - 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float sn = ec < half ? -s[i] : s[i], y = x[i] * c[i] + p[i] * sn;
    v[i] = ec < 2 * half ? y : x[i];
    v[i] = e < dk ? v[i] : 0.f;
  }
}

// retention_chunk for blockIdx.z: 128 key rows x 128 of the dv columns. A thread rotates four dimensions of eight tokens.
constexpr int PD = 128, PC = 128;
__global__ __launch_bounds__(NT, 2) void retention_chunk_parts_kernel(const bf16_t* __restrict__ p, int64_t stride, int H, int dk, int dv,
                                                                      Rot rot, const float* __restrict__ powers, int pw_stride,
                                                                      const int* __restrict__ c_start, int c0, float* __restrict__ c_state) {
  __shared__ __attribute__((aligned(16))) u32x4_t sK[3][8][PD], sV[8][PC];  // a piece: eight tokens of a dimension, of a column
  const int c = blockIdx.x, h = blockIdx.y, ncb = dv / PC;
  const int d0 = (int)(blockIdx.z / ncb) * PD, col0 = (int)(blockIdx.z % ncb) * PC;
  const int64_t t0 = c_start[c0 + c];
  const int n = c_start[c0 + c + 1] - (int)t0, half = rot.dims >> 1;
  const float kscale = 1.f / sqrtf((float)dk);
  const float* pw = powers + (int64_t)h * pw_stride;
  const bf16_t* keys = p + t0 * stride + (H + h) * dk;
  const bf16_t* vals = p + t0 * stride + 2 * H * dk + h * dv + col0;
  int64_t pos0;
  {
    const int g = threadIdx.x & 31, jg = threadIdx.x >> 5;
    uint32_t rows[8][2];
    load_v<4, false>(buffer(vals), stride, 4 * g, n, [&](int i) { return 8 * jg + i; }, rows);
    float w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = pw[max(n - 1 - (8 * jg + i), 0)];
    pos0 = rot.positions[t0];
    Raw4 raw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int jc = min(8 * jg + i, n - 1);
      raw[i] = load_raw(keys + jc * stride, d0 + 4 * g, dk, rot.cos_sin + (pos0 + jc) * rot.dims, half);
    }
    float k[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      rotate(raw[i], d0 + 4 * g, dk, half, k[i]);
#pragma unroll
      for (int x = 0; x < 4; ++x) k[i][x] = 8 * jg + i < n ? k[i][x] * (kscale * w[i]) : 0.f;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int at = place<4>(4 * g + x);
      sV[jg][at] = column<4>(rows, x);
      const float a[4] = {k[0][x], k[1][x], k[2][x], k[3][x]}, b[4] = {k[4][x], k[5][x], k[6][x], k[7][x]};
      const Parts s = split_vals(a, b);
#pragma unroll
      for (int i = 0; i < 3; ++i) sK[i][jg][at] = s.p[i];
    }
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  f32x4_t acc[2][8] = {};  // columns 32 wave + 16 m + 4 kq .., dimension 16 b + r16
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (32 * t >= n) break;
    u32x4_t a[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) a[m] = sV[4 * t + kq][place<4>(32 * wave + 16 * m + r16)];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (d0 + 16 * b >= dk) break;
#pragma unroll
      for (int i = 2; i >= 0; --i) {
        const u32x4_t k = sK[i][4 * t + kq][place<4>(16 * b + r16)];
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[m][b] = mfma_bf(a[m], k, acc[m][b]);
      }
    }
  }
  float* dst = c_state + ((int64_t)c * H + h) * dk * dv + col0;
  bool bad = false;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int d = d0 + 16 * b + r16;
    if (d >= dk) break;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const f32x4_t v = acc[m][b] * UP1;
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= !(fabsf(v[e]) <= 3.4028235e38f);
      *reinterpret_cast<f32x4_t*>(dst + (int64_t)d * dv + 32 * wave + 16 * m + 4 * kq) = v;
    }
  }
  if (!__syncthreads_or(bad)) return;
  for (int e = threadIdx.x; e < PD * PC; e += NT) {
    const int d = d0 + e / PC, col = e % PC;
    if (d >= dk) break;
    float s = 0.f;
    for (int j = 0; j < n; ++j)
      s += rot1(keys + j * stride, d, rot.cos_sin + (pos0 + j) * rot.dims, half) * (kscale * pw[n - 1 - j]) * ld(vals + j * stride + col);
    dst[(int64_t)d * dv + col] = s;
  }
}

// retention_out for heads of 32 NKD dimensions and 16 NCB columns: all keys are rotated and split at once (their loads fly together), then
// the weights' product with the values, then the state's, 32 dimensions x 128 columns at a time in two buffers, two pieces ahead in registers.
template <int NKD, int NCB>
__global__ __launch_bounds__(NT, 3) void retention_out_parts_kernel(const bf16_t* __restrict__ p, int64_t stride, int H, int gate, Rot rot,
                                                                    const float* __restrict__ powers, int pw_stride, float eps,
                                                                    const int* __restrict__ c_start, int c0,
                                                                    const float* __restrict__ c_state, bf16_t* __restrict__ out) {
  constexpr int dk = 32 * NKD, dv = 16 * NCB, NH = dv / 128, W = NCB / 4;  // W: columns of a thread where values are staged
  constexpr int KS = C + 2;                                                // pieces of a lane group's keys, and two: banks of their own
  constexpr int PIECE = 3 * 4 * 128, PIECES = NKD * NH;
  constexpr int LDS = std::max(3 * NKD * 4 * KS, std::max(2 * 4 * dv, 2 * PIECE));
  __shared__ __attribute__((aligned(16))) u32x4_t sL[LDS];
  __shared__ float sP[C + 1], red[NT / 64];
  static_assert(C * C * 4 <= (int)sizeof(sL) && PIECES >= 2, "");
  const int c = blockIdx.x, h = blockIdx.y;
  const int64_t t0 = c_start[c0 + c];
  const int n = c_start[c0 + c + 1] - (int)t0, half = rot.dims >> 1;
  const float kscale = 1.f / sqrtf((float)dk);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  if (threadIdx.x <= C) sP[threadIdx.x] = powers[(int64_t)h * pw_stride + threadIdx.x];
  const float* S0 = c_state + ((int64_t)c * H + h) * dk * dv;
  const int64_t pos0 = rot.positions[t0];
  const bf16_t* keys = p + t0 * stride + (H + h) * dk;
  const bf16_t* vals = p + t0 * stride + 2 * H * dk + h * dv;
  const int qi = wave * 16 + r16, qc = min(qi, n - 1), kj = threadIdx.x >> 2, kc = min(kj, n - 1), ks = threadIdx.x & 3;
  float q[NKD][8];  // this lane's query, dimensions 32 pc + 8 kq ..
  {
    Raw4 raw[NKD][2];
    const bf16_t* row = p + (t0 + qc) * stride + h * dk;
    const float* cs = rot.cos_sin + (pos0 + qc) * rot.dims;
#pragma unroll
    for (int pc = 0; pc < NKD; ++pc)
#pragma unroll
      for (int x = 0; x < 2; ++x) raw[pc][x] = load_raw(row, 32 * pc + 8 * kq + 4 * x, dk, cs, half);
#pragma unroll
    for (int pc = 0; pc < NKD; ++pc)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        float v[4];
        rotate(raw[pc][x], 32 * pc + 8 * kq + 4 * x, dk, half, v);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[pc][4 * x + i] = v[i];
      }
  }
  const auto query = [&](int pc) {
    const float a[4] = {q[pc][0], q[pc][1], q[pc][2], q[pc][3]}, b[4] = {q[pc][4], q[pc][5], q[pc][6], q[pc][7]};
    return split_vals(a, b);
  };
  {
    Raw4 raw[NKD][2];
    const float* cs = rot.cos_sin + (pos0 + kc) * rot.dims;
#pragma unroll
    for (int pc = 0; pc < NKD; ++pc)
#pragma unroll
      for (int x = 0; x < 2; ++x) raw[pc][x] = load_raw(keys + kc * stride, 32 * pc + 8 * ks + 4 * x, dk, cs, half);
#pragma unroll
    for (int pc = 0; pc < NKD; ++pc) {
      float a[4], b[4];
      rotate(raw[pc][0], 32 * pc + 8 * ks, dk, half, a);
      rotate(raw[pc][1], 32 * pc + 8 * ks + 4, dk, half, b);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] *= kscale, b[i] *= kscale;
      const Parts kp = split_vals(a, b);
#pragma unroll
      for (int i = 0; i < 3; ++i) sL[((i * NKD + pc) * 4 + ks) * KS + kj] = kp.p[i];
    }
  }
  const __amdgpu_buffer_rsrc_t rs = buffer(S0), rv = buffer(vals);
  uint32_t rows[2][8][W / 2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
    load_v<W, true>(rv, stride, W * lane, n, [&](int i) { return 32 * t + 16 * (i >> 2) + 4 * wave + (i & 3); }, rows[t]);
  __syncthreads();
  f32x4_t o[NCB], w[4];  // o[m][r]: column 16 m + 4 kq + r of query r16 of the wave; w[jb][r]: key 16 jb + 4 kq + r of that query
#pragma unroll
  for (int m = 0; m < NCB; ++m) o[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) w[jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int pc = 0; pc < NKD; ++pc) {
    const Parts qp = query(pc);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) {
      if (jb > wave) break;  // keys after every query of this wave
      u32x4_t f[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) f[i] = sL[((i * NKD + pc) * 4 + kq) * KS + 16 * jb + r16];
      w[jb] = mfma_six(f, qp.p, w[jb]);
    }
  }
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int dist = qi - (jb * 16 + kq * 4 + r);
      w[jb][r] = dist >= 0 ? w[jb][r] * moe_tile::SPLIT_DOWN * sP[max(dist, 0)] : 0.f;
    }
  __syncthreads();  // the keys are read
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int x = 0; x < W; ++x) sL[(4 * t + wave) * dv + place<W>(W * lane + x)] = column<W>(rows[t], x);
  float2 s[2][8];  // eight dimensions of two columns, of the next two pieces
  const auto load_s = [&](int piece) {
    const int src = ((piece / NH * 32 + 8 * wave) * dv + piece % NH * 128) * 4;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s[piece & 1][i] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, 8 * lane, src + i * dv * 4, 0));
  };
  load_s(0);
  load_s(1);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (2 * t > wave) break;
    const float lo[4] = {w[2 * t][0], w[2 * t][1], w[2 * t][2], w[2 * t][3]}, hi[4] = {w[2 * t + 1][0], w[2 * t + 1][1], w[2 * t + 1][2], w[2 * t + 1][3]};
    const Parts wp = split_vals(lo, hi);
#pragma unroll
    for (int m = 0; m < NCB; ++m) {
      const u32x4_t f = sL[(4 * t + kq) * dv + place<W>(16 * m + r16)];
#pragma unroll
      for (int i = 2; i >= 0; --i) o[m] = mfma_bf(f, wp.p[i], o[m]);
    }
  }
  // the state's part: the row's decay goes into its query; sums times 2^48 like the products that follow
#pragma unroll
  for (int m = 0; m < NCB; ++m) o[m] *= 1.f / UP1;
  const float decay = sP[qi + 1];
#pragma unroll
  for (int pc = 0; pc < NKD; ++pc)
#pragma unroll
    for (int i = 0; i < 8; ++i) q[pc][i] *= decay;
  __syncthreads();  // the values are read
  uint2 g[NCB] = {};
  Parts qp;
#pragma unroll
  for (int piece = 0; piece < PIECES; ++piece) {
    u32x4_t* buf = sL + (piece & 1) * PIECE;  // (read two pieces ago, with a barrier since)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      float u[4], v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = x ? s[piece & 1][i].y : s[piece & 1][i].x, v[i] = x ? s[piece & 1][4 + i].y : s[piece & 1][4 + i].x;
      const Parts sp = split_vals(u, v);
#pragma unroll
      for (int i = 0; i < 3; ++i) buf[(4 * i + wave) * 128 + place<2>(2 * lane + x)] = sp.p[i];
    }
    if (piece + 2 < PIECES) load_s(piece + 2);
    if (piece + 1 == PIECES && gate) {
      const bf16_t* grow = p + (t0 + qc) * stride + 2 * H * dk + H * dv + h * dv;
#pragma unroll
      for (int m = 0; m < NCB; ++m) g[m] = *reinterpret_cast<const uint2*>(grow + 16 * m + 4 * kq);
    }
    if (piece % NH == 0) qp = query(piece / NH);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      u32x4_t f[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) f[i] = buf[(4 * i + kq) * 128 + place<2>(16 * m + r16)];
      o[piece % NH * 8 + m] = mfma_six(f, qp.p, o[piece % NH * 8 + m]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int m = 0; m < NCB; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[m][r] *= moe_tile::SPLIT_DOWN;
      ss += o[m][r] * o[m][r];
    }
  ss = row_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)dv + eps);
  if (qi < n) {
    bf16_t* row = out + ((t0 + qi) * H + h) * dv;
#pragma unroll
    for (int m = 0; m < NCB; ++m) {
      if (gate) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[m][r] *= Fn<bf16_t>::silu(__uint_as_float(r & 1 ? (r < 2 ? g[m].x : g[m].y) & 0xffff0000u : (r < 2 ? g[m].x : g[m].y) << 16));
      }
      bf16_t v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) st(&v[r], o[m][r] * inv);
      *reinterpret_cast<uint2*>(row + 16 * m + 4 * kq) = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
    }
  }
  if (!__syncthreads_or(qi < n && !(ss <= 3.4028235e38f))) return;
  float* sW = reinterpret_cast<float*>(sL);
  for (int e = threadIdx.x; e < n * C; e += NT) {
    const int i = e / C, j = e % C;
    float a = 0.f;
    if (j <= i)
      for (int d = 0; d < dk; ++d)
        a += rot1(p + (t0 + i) * stride + h * dk, d, rot.cos_sin + (pos0 + i) * rot.dims, half) *
             (rot1(keys + j * stride, d, rot.cos_sin + (pos0 + j) * rot.dims, half) * kscale);
    sW[e] = j <= i ? a * sP[i - j] : 0.f;
  }
  __syncthreads();
  for (int i = 0; i < n; ++i) {
    const int col = min((int)threadIdx.x, dv - 1);
    const int64_t t = t0 + i;
    float a = 0.f;
    for (int d = 0; d < dk; ++d)
      a += rot1(p + t * stride + h * dk, d, rot.cos_sin + (pos0 + i) * rot.dims, half) * S0[(int64_t)d * dv + col];
    a *= sP[i + 1];
    for (int j = 0; j <= i; ++j) a += sW[i * C + j] * ld(vals + j * stride + col);
    const float norm = 1.f / sqrtf(block_sum<NT>((int)threadIdx.x < dv ? a * a : 0.f, red) / (float)dv + eps);
    if (gate) a *= Fn<bf16_t>::silu(ld(p + t * stride + 2 * H * dk + H * dv + h * dv + col));
    if ((int)threadIdx.x < dv) st(out + (t * H + h) * dv + col, a * norm);
  }
}

template <typename T>
int launch(const T* p, int64_t stride, int H, int dk, int dv, int gate, const Rot& rot, const float* powers, int pw_stride,
           float eps, float* state, const int* seq_start, const int* seq_slot, const int* seq_init, T* out, int T_rows,
           int nseq, int nd, int nc, const int* c_start, const int* s_chunk0, float* c_state, float* o_raw,
           hipStream_t stream) {
  constexpr size_t es = sizeof(T);
  if (nd > 0) {
    const bool v4 = dv % 4 == 0 && ((uintptr_t)state & 15) == 0;
    const int cols = v4 ? dv / 4 : dv, ncg = std::min(cols, NT), RG = std::min(NT / ncg, dk);
    const size_t lds = (size_t)(2 * dk + RG * dv) * sizeof(float);
    if (lds > 64 * 1024) return 1;
    const dim3 grid(H, nd);
    if (v4)
      hipLaunchKernelGGL((retention_step_kernel<T, 4>), grid, dim3(NT), lds, stream, p, stride, H, dk, dv, gate, rot,
                         powers, pw_stride, eps, state, seq_start, seq_slot, seq_init, out, ncg, RG);
    else
      hipLaunchKernelGGL((retention_step_kernel<T, 1>), grid, dim3(NT), lds, stream, p, stride, H, dk, dv, gate, rot,
                         powers, pw_stride, eps, state, seq_start, seq_slot, seq_init, out, ncg, RG);
  }
  if (nd >= nseq) return 0;
  const int n = nc - nd;  // chunks of the longer runs
  // 16-byte pieces of the state, four elements of a projection row at a time
  const bool vec = dk % 4 == 0 && dv % 4 == 0 && (rot.dims >> 1) % 4 == 0 && stride % 4 == 0 &&
                   ((uintptr_t)p & (4 * es - 1)) == 0 && ((uintptr_t)rot.cos_sin & 15) == 0;
  auto set = [](const void* k, size_t lds) {
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  };
#define SM_CHUNK(NCB, VEC)                                                                                            \
  {                                                                                                                   \
    const size_t lds = (size_t)(C * QS + C * (16 * NCB + 4)) * sizeof(float);                                         \
    const dim3 grid(n, H, ((dk + DB - 1) / DB) * ((dv + 16 * NCB - 1) / (16 * NCB)));                                 \
    set((const void*)retention_chunk_kernel<T, NCB, VEC>, lds);                                                       \
    hipLaunchKernelGGL((retention_chunk_kernel<T, NCB, VEC>), grid, dim3(NT), lds, stream, p, stride, H, dk, dv, rot, \
                       powers, pw_stride, c_start, nd, c_state);                                                      \
  }
  // bf16 rows on the bf16 units. Heads of 64 or 128 x 128 or 256, whose keys fit three workgroups' LDS on a CU; rows whose 64 tokens lie within
  // 31 bits
  bool parts = false;
  Rot any = rot;  // without a rotation the loads of its table go somewhere
  if (rot.dims == 0) any.cos_sin = powers;
  if constexpr (es == 2) {
    parts = vec && stride <= 1 << 23 && (dk == 64 || dk == 128) && (dv == 128 || dv == 256) && ((uintptr_t)c_state & 15) == 0 &&
            ((uintptr_t)out & 7) == 0 && H * pw_stride >= 4;
    if (parts)
      hipLaunchKernelGGL(retention_chunk_parts_kernel, dim3(n, H, (dk + PD - 1) / PD * (dv / PC)), dim3(NT), 0, stream, p, stride, H, dk, dv, any,
                         powers, pw_stride, c_start, nd, c_state);
  }
  if (parts) {
  } else if (dv <= 64 && vec) SM_CHUNK(4, true)
  else if (dv <= 64) SM_CHUNK(4, false)
  else if (vec) SM_CHUNK(8, true)
  else SM_CHUNK(8, false)
#undef SM_CHUNK
  const int64_t per_head = (int64_t)dk * dv;
  // 16-byte pieces when that still leaves enough threads to fill the chip
  if (per_head % 4 == 0 && per_head * H * (nseq - nd) >= (int64_t)4 * 65536 && ((uintptr_t)state & 15) == 0 &&
      ((uintptr_t)c_state & 15) == 0)
    hipLaunchKernelGGL((retention_link_kernel<4>), dim3((unsigned)((per_head * H / 4 + NT - 1) / NT), nseq - nd), dim3(NT),
                       0, stream, c_state, c_start, s_chunk0, nd, nd, H, per_head, powers, pw_stride, state, seq_slot,
                       seq_init);
  else
    hipLaunchKernelGGL((retention_link_kernel<1>), dim3((unsigned)((per_head * H + NT - 1) / NT), nseq - nd), dim3(NT), 0,
                       stream, c_state, c_start, s_chunk0, nd, nd, H, per_head, powers, pw_stride, state, seq_slot,
                       seq_init);
  if constexpr (es == 2) {
    if (parts) {
      const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(n, H), dim3(NT), 0, stream, p, stride, H, gate, any, powers, pw_stride, eps, c_start, nd, c_state, out);
      };
      if (dk == 64 && dv == 128) go(retention_out_parts_kernel<2, 8>);
      else if (dk == 64) go(retention_out_parts_kernel<2, 16>);
      else if (dv == 128) go(retention_out_parts_kernel<4, 8>);
      else go(retention_out_parts_kernel<4, 16>);
      return 0;
    }
  }
#define SM_OUT(NCB, VEC)                                                                                              \
  {                                                                                                                   \
    const size_t lds = (size_t)(C * OS + OB * (16 * NCB + 4)) * sizeof(float);                                        \
    const dim3 grid(n, H, (dv + 16 * NCB - 1) / (16 * NCB));                                                          \
    set((const void*)retention_out_kernel<T, NCB, VEC>, lds);                                                         \
    hipLaunchKernelGGL((retention_out_kernel<T, NCB, VEC>), grid, dim3(NT), lds, stream, p, stride, H, dk, dv, gate,  \
                       rot, powers, pw_stride, eps, c_start, nd, c_state, out, o_raw);                                \
  }
#define SM_OUT2(VEC)                  \
  if (dv <= 64) SM_OUT(4, VEC)        \
  else if (dv <= 128) SM_OUT(8, VEC)  \
  else SM_OUT(16, VEC)
  if (vec) { SM_OUT2(true) }
  else { SM_OUT2(false) }
#undef SM_OUT2
#undef SM_OUT
  if (o_raw != nullptr) {
    const int rows = T_rows - nd;  // the longer runs' tokens follow the nd single ones
    hipLaunchKernelGGL((retention_norm_kernel<T>), dim3(rows, std::max(1, std::min((H + 3) / 4, 4096 / rows))), dim3(NT), 0,
                       stream, o_raw, p, stride, H, dk, dv, gate, eps, c_start + nd, out);
  }
  return 0;
}

}  // namespace

extern "C" {

int sm_retention_chunk() { return C; }
int sm_retention_cols() { return MAXCOLS; }

// The first nd sequences bring one token each; the chunks of the others are numbers nd .. nc - 1 of c_start [nc + 1],
// s_chunk0 [nseq + 1] bounds each sequence's chunks. Workspaces (fp32): c_state [nc - nd, H, dk, dv]; o_raw
// [T, H, dv] when dv > sm_retention_cols(), else null. Returns 0, or 1 when the sizes do not fit.
int sm_retention(const void* p, int64_t stride, int H, int dk, int dv, int gate, const int64_t* positions,
                 const float* cos_sin, int rot_dims, const float* powers, int pw_stride, float eps, float* state,
                 const int* seq_start, const int* seq_slot, const int* seq_init, void* out, int T, int nseq, int nd,
                 int f32, int nc, const int* c_start, const int* s_chunk0, float* c_state, float* o_raw,
                 hipStream_t stream) {
  const Rot rot{positions, cos_sin, rot_dims};
  if (f32)
    return launch<float>((const float*)p, stride, H, dk, dv, gate, rot, powers, pw_stride, eps, state, seq_start, seq_slot,
                         seq_init, (float*)out, T, nseq, nd, nc, c_start, s_chunk0, c_state, o_raw, stream);
  return launch<bf16_t>((const bf16_t*)p, stride, H, dk, dv, gate, rot, powers, pw_stride, eps, state, seq_start, seq_slot,
                        seq_init, (bf16_t*)out, T, nseq, nd, nc, c_start, s_chunk0, c_state, o_raw, stream);
}

}  // extern "C"
