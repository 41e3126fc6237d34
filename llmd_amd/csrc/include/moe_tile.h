// Grouped expert GEMMs: sorting of (token, choice) pairs by expert, and the tile bodies on the matrix cores. Shared by the expert
// kernels of both op libraries, which bring the weight layout (wrow) and what happens to the sums (out).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "moe_sort.h"
#include <type_traits>
#include <utility>

namespace moe_tile {

// order (where it is asked for): the tiles by their number of 16-row blocks, most first. cnt, first: LDS, an expert's pairs and
// its first tile, written by this workgroup.
constexpr int SIZES = 8;  // blocks of 16 rows that a tile can have
__device__ __forceinline__ void by_size(const int* cnt, const int* first, int E, int tm, int* __restrict__ order, int* sizes) {
  const int tid = threadIdx.x;
  if (tid < SIZES) sizes[tid] = 0;
  __syncthreads();
  auto last = [&](int e) { return cnt[e] - (cnt[e] - 1) / tm * tm; };  // rows of an expert's last tile
  auto bin = [](int rows) { return SIZES - (rows + 15) / 16; };
  for (int e = tid; e < E; e += blockDim.x)
    if (cnt[e] > 0) {
      atomicAdd(&sizes[bin(last(e))], 1);
      if (cnt[e] > tm) atomicAdd(&sizes[bin(tm)], (cnt[e] - 1) / tm);
    }
  __syncthreads();
  if (tid == 0)
    for (int i = 0, at = 0; i < SIZES; ++i) {
      const int n = sizes[i];
      sizes[i] = at;
      at += n;
    }
  __syncthreads();
  for (int e = tid; e < E; e += blockDim.x)
    if (cnt[e] > 0) {
      const int full = (cnt[e] - 1) / tm;
      order[atomicAdd(&sizes[bin(last(e))], 1)] = first[e] + full;
      if (full > 0)
        for (int i = 0, at = atomicAdd(&sizes[bin(tm)], full); i < full; ++i) order[at + i] = first[e] + i;
    }
}

// Sorts the pairs by expert into tiles of ``tm`` slots. tiles[0] = number of tiles, then for each tile three numbers:
// expert | rows << 16 (the tile's first ``rows`` slots hold pairs, slot_row says which), its expert's first tile and number
// of tiles. A pair's rank inside its expert is what its LDS counter
// returned (kept in pair_slot between the passes), so the pairs are counted once; the experts' first tiles come from one
// scan over the workgroup. 512 pairs over 128 experts: 13.7 us with a serial scan by one thread and all slots marked, now 4 us.
__global__ __launch_bounds__(1024) static void moe_group_kernel(const int* __restrict__ ids, int n, int E, int tm,
                                                         int* __restrict__ slot_row, int* __restrict__ tiles,
                                                         int* __restrict__ pair_slot, int* __restrict__ order) {
  extern __shared__ int sh[];  // cnt[E] | first tile[E]
  __shared__ int wsum[16], sizes[SIZES];
  int* cnt = sh;
  int* first = sh + E;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int p0 = 0; p0 < n; p0 += 1024 * 8) {
    int e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int p = p0 + i * 1024 + tid;
      e[i] = p < n ? ids[p] : E;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int p = p0 + i * 1024 + tid;
      if (p < n) pair_slot[p] = (unsigned)e[i] < (unsigned)E ? atomicAdd(&cnt[e[i]], 1) : -1;  // any other id: no tile, slot -1
    }
  }
  __syncthreads();
  // every thread owns ``per`` neighbouring experts
  const int per = (E + 1023) / 1024, e0 = tid * per;
  int mine = 0;
  for (int i = 0; i < per; ++i)
    if (e0 + i < E) mine += (cnt[e0 + i] + tm - 1) / tm;
  int scan = mine;  // inclusive over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(scan, o, 64);
    if (lane >= o) scan += v;
  }
  if (lane == 63) wsum[wave] = scan;
  __syncthreads();
  int at = scan - mine;
  for (int w = 0; w < wave; ++w) at += wsum[w];
  for (int j = 0; j < per; ++j) {
    const int e = e0 + j;
    if (e >= E) break;
    first[e] = at;
    const int nt = (cnt[e] + tm - 1) / tm;
    for (int i = 0, left = cnt[e]; i < nt; ++i, ++at, left -= tm) {
      tiles[1 + 3 * at] = e | (left < tm ? left : tm) << 16;
      tiles[2 + 3 * at] = first[e];
      tiles[3 + 3 * at] = nt;
    }
  }
  if (tid == 1023) tiles[0] = at;
  if (order != nullptr) by_size(cnt, first, E, tm, order, sizes);
  __syncthreads();
  for (int p0 = 0; p0 < n; p0 += 1024 * 8) {
    int r[8], e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int p = p0 + i * 1024 + tid;
      r[i] = p < n ? pair_slot[p] : -1;
      e[i] = p < n ? ids[p] : 0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int p = p0 + i * 1024 + tid;
      if (r[i] < 0) continue;
      const int slot = first[e[i]] * tm + r[i];
      slot_row[slot] = p;
      pair_slot[p] = slot;
    }
  }
}

// The same over many workgroups (moe_sort.h), pair_slot holding the ranks: 16384 pairs over 128 experts 18.5 -> 10 us.
__global__ __launch_bounds__(moe_sort::NT) static void moe_group_place_kernel(const int* __restrict__ ids, int n, int E, int tm,
                                                                              const int* __restrict__ hist,
                                                                              int* __restrict__ slot_row,
                                                                              int* __restrict__ tiles,
                                                                              int* __restrict__ pair_slot,
                                                                              int* __restrict__ order) {
  __shared__ int sizes[SIZES];
  extern __shared__ int sh[];  // pairs[E] | first tile[E] | pairs in the blocks before[E]
  int *cnt = sh, *first = sh + E;
  const int total = moe_sort::plan(hist, gridDim.x, E, tm, cnt, first, sh + 2 * E);
  if (blockIdx.x == 0 && threadIdx.x == 0) tiles[0] = total;
  // each block lists the tiles of its share of the experts
  for (int e = blockIdx.x + gridDim.x * threadIdx.x; e < E; e += gridDim.x * moe_sort::NT) {
    const int nt = (cnt[e] + tm - 1) / tm;
    for (int i = 0, left = cnt[e]; i < nt; ++i, left -= tm) {
      int* t = tiles + 1 + 3 * (first[e] + i);
      t[0] = e | (left < tm ? left : tm) << 16;
      t[1] = first[e];
      t[2] = nt;
    }
  }
  if (order != nullptr && blockIdx.x == 0) by_size(cnt, first, E, tm, order, sizes);
  moe_sort::place(ids, n, tm, first, sh + 2 * E, slot_row, pair_slot);
}

// ``hist`` (blocks(n) * E numbers): where moe_sort::many(n, E).
static inline void launch_group(const int* ids, int n, int E, int tm, int* hist, int* slot_row, int* tiles, int* pair_slot,
                                int* order, hipStream_t stream) {
  if (!moe_sort::many(n, E)) {
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), 2 * E * sizeof(int), stream, ids, n, E, tm, slot_row, tiles,
                       pair_slot, order);
    return;
  }
  const dim3 grid(moe_sort::blocks(n)), wg(moe_sort::NT);
  hipLaunchKernelGGL(moe_sort::moe_count_kernel, grid, wg, E * sizeof(int), stream, ids, n, E, pair_slot, hist);
  hipLaunchKernelGGL(moe_group_place_kernel, grid, wg, 3 * E * sizeof(int), stream, ids, n, E, tm, hist, slot_row, tiles,
                     pair_slot, order);
}

// On the matrix cores, both types: a workgroup owns one tile (up to 128 rows of one expert) and 128 weight rows.
// bf16: v_mfma_f32_16x16x32_bf16; fp32: the same on three parts of every number (moe_tile_split below), and for rows with infinities
// and NaNs v_mfma_f32_16x16x4_f32 on the same 16-byte pieces (element j of a lane's piece belongs
// to product j, in both operands alike). Weights are the products' A operand: a lane ends up with four neighbouring columns of
// one row. fp32 accumulation in a fixed order of K: a row's sums do not depend on its tile. Loads run PD steps of 128 bytes
// per row ahead of the products, in registers; LDS has two buffers and one barrier per step.
//   up to 32 rows : nothing but the weights' stream counts. Each wave takes 32 weight rows straight into the registers that
//                   the products read; only the activations pass LDS. (A quarter of a wave then touches 16 rows, which the
//                   vector cache serves at 16 bytes per clock: above HBM's rate, but not above that of weights shared by
//                   several tiles.)
//   more rows     : weights pass LDS too, read from memory a whole 128-byte line per eight lanes. Up to 64 rows the waves
//                   split the weight rows, beyond that two by two in bf16, where the reads of LDS count. In fp32 the products
//                   and the splitting do: there the waves split the weight rows up to the end, and a tile costs
//                   its blocks of 16 rows, not 128.
// 128 gated experts of 2048 x 768, first + second product, us. bf16, 512 rows: 64 x 128 tiles through one LDS buffer 147 + 82,
// this 138 + 73 (5.7 and 5.4 TB/s of weights). fp32, 5600 rows by a skewed router: FMA form 1707 + 905, fp32 instructions 412 + 210, this 365 + 185.
//
// Work items are (expert, block of weight rows, tile), the tiles of one block side by side: they read the same weights at the
// same time, once from memory (tile by tile, an expert's second tile came too late for L2: 1.65 GB for 0.8 GB of weights at
// 32768 rows). The list is cut into eight ranges, one per XCD, so that an XCD's workgroups share an expert's rows too.
// In fp32, from 16 rows per expert on, the tiles' products differ more than their weights' streams, and the XCDs' ranges with them:
// the tiles go to the XCDs in turn, those with the most rows first (find_work_by_size). 128 gated experts of 2048 x 768, 8 chosen,
// by a skewed router (700 tokens: 4 to 126 rows), both products with sorting and sum, us, fp32 instructions, before / rows by 16 / and by size:
// 700 tokens 838 / 751 / 653, 1400 1380 / 1256 / 1020, 2048 1782 / 1701 / 1394 (118 of the 152 TFLOP/s that a large product
// reaches). The line: by expert / by size at 17, 19, 22, 28, 36 rows per expert, uniform router 482 / 478, 466 / 486, 485 / 494,
// 522 / 518, 598 / 577, skewed 598 / 505, 517 / 510, 706 / 549, 778 / 577, 921 / 645; 4 rows 436 / 458. Largest and smallest in turn,
// so that one's products pass beside the other's weights: 665, 1037, 1449. Three steps of loads ahead instead of two: equal.
// Gated forms: the 128 weight rows are 64 gate columns and the matching up columns.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <typename T> __device__ __forceinline__ void mma16(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b);
template <> __device__ __forceinline__ void mma16<uint16_t>(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}
template <> __device__ __forceinline__ void mma16<float>(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
  const f32x4_t x = __builtin_bit_cast(f32x4_t, a), y = __builtin_bit_cast(f32x4_t, b);
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], y[j], acc, 0, 0, 0);
}

struct MoeTile {  // what the bodies below share
  int K;
  char* lds;
  const char* w;      // the expert's weights; wrow(j) below: byte offset of the tile's weight row j
  const char* ap[4];  // this thread's pieces of the rows: row (tid >> 3) + 32 i, bytes (tid & 7) * 16 of a step
};

// what this wave has written is in LDS and all waves have arrived; loads stay in flight (a __syncthreads would drain them)
__device__ __forceinline__ void meet() {
  __builtin_amdgcn_sched_barrier(0);  // and steps stay apart: moved into one another they need more registers than there are
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Rows of an LDS buffer are 128 bytes; piece c of row r lies at place c ^ (r / 2 mod 8): the 16 rows that a quarter of a wave
// reads, and the two rows that it writes, then take all 64 banks.
constexpr int TLS = 128;
__device__ __forceinline__ int lds_wr(int tid) { return (tid >> 3) * TLS + ((tid ^ tid >> 4) & 7) * 16; }
__device__ __forceinline__ int lds_rd(int r16, int kq) { return r16 * TLS + ((kq ^ r16 >> 1) & 7) * 16; }  // ^ 64: pieces 4 .. 7
constexpr int TBM = 128, TBW = 128;    // rows and weight rows of a tile
constexpr int TBUF = TBM * TLS;        // bytes of one operand's buffer

// Drives the steps of K: first(s) starts the loads of step s, step(s, kt, next, first_operand, second_operand) is step kt
// whose registers are set s = kt % PD; the flags (types) say whether a step follows, whether kt + 1 + PD exists and
// whether kt + PD does. The long part has every load in every step and the last R steps are spelled out for
// each remainder: behind a load under a condition hipcc can only wait for all loads in flight.
template <bool B> using Flag = std::integral_constant<bool, B>;
template <int S> using Set = std::integral_constant<int, S>;

template <int PD, int R, typename Step, int... J>
__device__ __forceinline__ void last_steps(int nk, Step& step, std::integer_sequence<int, J...>) {
  (step(Set<J % PD>{}, nk - R + J, Flag<(J + 1 < R)>{}, Flag<(J + 1 + PD < R)>{}, Flag<(J + PD < R)>{}), ...);
}
template <int PD, typename Step, int... J>
__device__ __forceinline__ void full_steps(int k0, Step& step, std::integer_sequence<int, J...>) {
  (step(Set<J>{}, k0 + J, Flag<true>{}, Flag<true>{}, Flag<true>{}), ...);
}
template <int PD, typename First, typename Step, typename Begin>
__device__ __forceinline__ void k_steps(int nk, First first, Begin begin, Step step) {
  static_assert(PD == 2 || PD == 3, "the remainders below");
  if (nk > PD) {
#pragma unroll
    for (int s = 0; s < PD; ++s) first(s);
    begin(Flag<true>{});
    const int ns = (nk - 1 - PD) / PD * PD;
    for (int k0 = 0; k0 < ns; k0 += PD) full_steps<PD>(k0, step, std::make_integer_sequence<int, PD>{});
    const int left = nk - ns;  // PD + 1 .. 2 PD
    if (left == PD + 1) last_steps<PD, PD + 1>(nk, step, std::make_integer_sequence<int, PD + 1>{});
    else if (left == PD + 2) last_steps<PD, PD + 2>(nk, step, std::make_integer_sequence<int, PD + 2>{});
    else if (PD == 3) last_steps<PD, 2 * PD>(nk, step, std::make_integer_sequence<int, 2 * PD>{});
  } else if (nk > 0) {
#pragma unroll
    for (int s = 0; s < PD; ++s)
      if (s < nk) first(s);
    begin(Flag<false>{});
    if (nk == 1) last_steps<PD, 1>(nk, step, std::make_integer_sequence<int, 1>{});
    else if (nk == 2) last_steps<PD, 2>(nk, step, std::make_integer_sequence<int, 2>{});
    else last_steps<PD, 3>(nk, step, std::make_integer_sequence<int, 3>{});
  }
}

// Up to 16 MI rows (MI 1 or 2): weights straight to registers.
template <typename T, bool GATED, int MI, int PD, typename WRow, typename Out>
__device__ __forceinline__ void moe_tile_few(const MoeTile& t, WRow wrow, Out out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  const int kb = t.K * (int)sizeof(T), nk = kb >> 7;  // bytes of a row, whole steps
  const int wr = lds_wr(tid), rd = lds_rd(r16, kq);
  // weight rows of the wave: gated 16 gate rows and their up rows, else 32 neighbours
  uint32_t wp[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) wp[c] = wrow(GATED ? c * 64 + wave * 16 + r16 : wave * 32 + c * 16 + r16) + kq * 16;
  f32x4_t acc[2][MI];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[c][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wb[PD][2][2], ab[PD];
  auto load_a = [&](int s, int kt) { ab[s] = *reinterpret_cast<const u32x4_t*>(t.ap[0] + kt * 128); };
  auto load_w = [&](int s, int kt) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) wb[s][c][h] = *reinterpret_cast<const u32x4_t*>(t.w + kt * 128 + h * 64 + wp[c]);
  };
  auto store_a = [&](int s, int buf) { *reinterpret_cast<u32x4_t*>(t.lds + buf * TBUF + wr) = ab[s]; };
  auto products = [&](int s, int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const u32x4_t a = *reinterpret_cast<const u32x4_t*>(t.lds + ((buf * TBUF + rd + i * 16 * TLS) ^ (h * 64)));
#pragma unroll
        for (int c = 0; c < 2; ++c) mma16<T>(acc[c][i], wb[s][c][h], a);
      }
  };
  k_steps<PD>(
      nk,
      [&](int s) {
        load_a(s, s);
        load_w(s, s);
      },
      [&](auto more) {
        store_a(0, 0);
        if constexpr (more) load_a(0, PD);
      },
      [&](auto s, int kt, auto next, auto more_a, auto more_w) {
        meet();  // buffer kt & 1 is written, the other one read
        if constexpr (next) {
          store_a((s + 1) % PD, (kt + 1) & 1);
          if constexpr (more_a) load_a((s + 1) % PD, kt + 1 + PD);
        }
        products(s, kt & 1);
        if constexpr (more_w) load_w(s, kt + PD);
      });
  if (kb & 127) {  // the rest of K, a multiple of 16 bytes: pieces past the end are zeros
    const int left = kb & 127;
    const u32x4_t zero = {0, 0, 0, 0};
    ab[0] = (tid & 7) * 16 < left ? *reinterpret_cast<const u32x4_t*>(t.ap[0] + nk * 128) : zero;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wb[0][c][h] = kq * 16 + h * 64 < left ? *reinterpret_cast<const u32x4_t*>(t.w + nk * 128 + h * 64 + wp[c]) : zero;
    meet();
    store_a(0, 0);
    meet();
    products(0, 0);
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int c = 0; c < (GATED ? 1 : 2); ++c)
      out(i * 16 + r16, GATED ? wave * 16 + kq * 4 : wave * 32 + c * 16 + kq * 4, acc[c][i], acc[1][i]);
}

// More rows: both operands through LDS. WM waves share the rows, 4 / WM the weight rows; a wave has MI blocks of 16 rows.
template <typename T, bool GATED, int MI, int WM, int PD, typename WRow, typename Out>
__device__ __forceinline__ void moe_tile_many(const MoeTile& t, WRow wrow, Out out) {
  constexpr int NC = 2 * WM, NA = (MI * WM + 1) / 2;  // blocks of 16 weight rows per wave; pieces of the rows per thread and step
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  const int kb = t.K * (int)sizeof(T), nk = kb >> 7;
  const int wr = lds_wr(tid), ra = wm * MI * 16 * TLS + lds_rd(r16, kq);
  // gated: blocks 0 .. NC / 2 - 1 are gate rows, the others the matching up rows
  int rw[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
    rw[c] = 2 * TBUF + (GATED ? (c % (NC / 2)) * 16 + wn * 8 * NC + (c / (NC / 2)) * 64 : wn * 16 * NC + c * 16) * TLS + lds_rd(r16, kq);
  uint32_t wp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wp[i] = wrow((tid >> 3) + 32 * i) + (tid & 7) * 16;
  f32x4_t acc[NC][MI];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[c][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wb[PD][4], ab[PD][NA];
  auto load = [&](int s, int kt) {
#pragma unroll
    for (int i = 0; i < NA; ++i) ab[s][i] = *reinterpret_cast<const u32x4_t*>(t.ap[i] + kt * 128);
#pragma unroll
    for (int i = 0; i < 4; ++i) wb[s][i] = *reinterpret_cast<const u32x4_t*>(t.w + kt * 128 + wp[i]);
  };
  auto store = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) *reinterpret_cast<u32x4_t*>(t.lds + buf * TBUF + wr + i * 32 * TLS) = ab[s][i];
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4_t*>(t.lds + (2 + buf) * TBUF + wr + i * 32 * TLS) = wb[s][i];
  };
  auto products = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __builtin_amdgcn_sched_barrier(0);  // one half's pieces in registers at a time
      u32x4_t w[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) w[c] = *reinterpret_cast<const u32x4_t*>(t.lds + ((buf * TBUF + rw[c]) ^ (h * 64)));
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const u32x4_t a = *reinterpret_cast<const u32x4_t*>(t.lds + ((buf * TBUF + ra + i * 16 * TLS) ^ (h * 64)));
#pragma unroll
        for (int c = 0; c < NC; ++c) mma16<T>(acc[c][i], w[c], a);
      }
    }
  };
  k_steps<PD>(
      nk, [&](int s) { load(s, s); },
      [&](auto more) {
        store(0, 0);
        if constexpr (more) load(0, PD);
      },
      [&](auto s, int kt, auto next, auto more, auto) {
        meet();  // buffer kt & 1 is written, the other one read
        if constexpr (next) {
          store((s + 1) % PD, (kt + 1) & 1);
          if constexpr (more) load((s + 1) % PD, kt + 1 + PD);
        }
        products(kt & 1);
      });
  if (kb & 127) {  // as above
    const bool in = (tid & 7) * 16 < (kb & 127);
    const u32x4_t zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NA; ++i) ab[0][i] = in ? *reinterpret_cast<const u32x4_t*>(t.ap[i] + nk * 128) : zero;
#pragma unroll
    for (int i = 0; i < 4; ++i) wb[0][i] = in ? *reinterpret_cast<const u32x4_t*>(t.w + nk * 128 + wp[i]) : zero;
    meet();
    store(0, 0);
    meet();
    products(0);
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int c = 0; c < (GATED ? NC / 2 : NC); ++c)
      out((wm * MI + i) * 16 + r16, (GATED ? wn * 8 * NC : wn * 16 * NC) + c * 16 + kq * 4, acc[c][i], acc[(c + NC / 2) % NC][i]);
}

// fp32 on the bf16 units: a number is the sum of three bf16 parts (8 bits of its 24 each, rounded to nearest: exact), and the six
// largest products of parts are formed, in fp32 sums: a second part is at most 2^-8 of its number and a third 2^-17, so that each of the
// two largest products left out is at most 2^-25 of the whole. Numbers are taken times 2^24 and sums times 2^-48: the last bit of the
// smallest fp32 number, 2^-149, is then a normal bf16 number too (as they are, numbers of 2^-116
// give sums 2e-6 off and numbers of 2^-132 0.14). Numbers from 2^104 and sums from 2^80 on overflow so and are done again like infinities.
// Six 16 x 16 x 32 instructions of 16 cycles for what takes eight of 32 cycles in 16 x 16 x 4 fp32, beside 6.5 vector instructions per number split. Both products with sorting and sum of 128
// gated experts of 2048 x 768 with as many rows each, us, fp32 instructions / parts: 1 row 427 / 434, 16 453 / 449, 32 514 / 493, 44
// 590 / 524, 64 705 / 580, 80 835 / 660, 120 1240 / 940 (up to 64 rows the weights' stream counts, 414 us at its best); by a
// skewed router, 700 tokens 631 / 556, 1400 1002 / 805, 2048 1364 / 1072. Off 64 bits, relative: (2048, 768) 1.20e-6 / 1.03e-6, (4096, 2048)
// 1.75e-6 / 1.53e-6, (1000, 500) 8.7e-7 / 7.4e-7 (fewer roundings of the sums).
// The scaling is in none of these times: 128 rows of 8 chosen 327 / 330 us, 700 tokens 576 / 581, 2048 1118 / 1148.
struct Parts {
  u32x4_t p[3];  // 8 elements: largest part first
};
constexpr float SPLIT_UP = 0x1p24f, SPLIT_DOWN = 0x1p-48f;
// part i of four elements to (lo, hi); x: what is left of them. (As vectors of two: hipcc rounds scalar casts twice, and does not keep
// the distance that the matrix units need from what asm writes.)
__device__ __forceinline__ void take_part(f32x4_t& x, uint32_t& lo, uint32_t& hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{x[0], x[1]}, bf16x2_t));
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{x[2], x[3]}, bf16x2_t));
  x[0] -= __uint_as_float(lo << 16), x[1] -= __uint_as_float(lo & 0xffff0000u);
  x[2] -= __uint_as_float(hi << 16), x[3] -= __uint_as_float(hi & 0xffff0000u);
}
__device__ __forceinline__ Parts split8(const u32x4_t& first, const u32x4_t& second) {
  f32x4_t x = __builtin_bit_cast(f32x4_t, first) * SPLIT_UP, y = __builtin_bit_cast(f32x4_t, second) * SPLIT_UP;
  Parts r;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    uint32_t a, b, c, d;
    take_part(x, a, b);
    take_part(y, c, d);
    r.p[i] = u32x4_t{a, b, c, d};
  }
  return r;
}

// fp32: rows as parts in LDS (split once), weights as they are, each wave splits its own. Up to 32 rows (DIRECT) the weights go straight to
// registers as in moe_tile_few, else through LDS. A lane's 8 of a step's 32 elements are pieces kq and kq + 4 of a row, in
// both operands. Every tile size sums in the same order: a row's bits do not depend on its tile.
// LDS: two buffers of 128 weight rows of 128 bytes, two of 3 parts x 128 rows x 64 bytes; piece q of 16 bytes of row r of a part at
// place q ^ F(r / 4 mod 4), F = 0 2 3 1. Parts of an infinite or NaN element, or of one that rounds to infinity, make NaNs of the
// sums that it belongs to: rows with a sum that is not finite are not put out; true if there are any (bit i of rows_left: row 16 i + this
// lane's).
constexpr int SROW = 64, SPART = TBM * SROW, SBUF = 3 * SPART;
constexpr int SLDS = 2 * TBUF + 2 * SBUF;  // 80 KB: two workgroups per CU
template <bool GATED, int MI, int PD, bool DIRECT, typename WRow, typename Out>
__device__ __forceinline__ bool moe_tile_split(const MoeTile& t, WRow wrow, Out out, uint32_t& rows_left) {
  constexpr int NA = (MI + 1) / 2;  // a thread's pieces of the rows in a step
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  const int kb = t.K * 4, nk = kb >> 7;
  const auto place = [](int row, int q) { return row * SROW + ((q ^ (0x1E >> (2 * (row >> 2 & 3)) & 3)) * 16); };
  const int wr = lds_wr(tid), sa = 2 * TBUF + place(tid >> 3, tid & 3) + (tid & 4) * 2, ra = 2 * TBUF + place(r16, kq);
  // the wave's weight rows: gated 16 gate rows and their up rows, else 32 neighbours
  const auto own = [&](int c) { return GATED ? c * 64 + wave * 16 : wave * 32 + c * 16; };
  uint32_t wp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    wp[i] = DIRECT ? wrow(own(i >> 1) + r16) + kq * 16 + (i & 1) * 64 : wrow((tid >> 3) + 32 * i) + (tid & 7) * 16;
  f32x4_t acc[2][MI];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[c][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wb[PD][4], ab[PD][NA];
  auto load_a = [&](int s, int kt) {
#pragma unroll
    for (int i = 0; i < NA; ++i) ab[s][i] = *reinterpret_cast<const u32x4_t*>(t.ap[i] + kt * 128);
  };
  auto load_w = [&](int s, int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) wb[s][i] = *reinterpret_cast<const u32x4_t*>(t.w + kt * 128 + wp[i]);
  };
  auto store = [&](int s, int buf) {
    if constexpr (!DIRECT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4_t*>(t.lds + buf * TBUF + wr + i * 32 * TLS) = wb[s][i];
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      f32x4_t x = __builtin_bit_cast(f32x4_t, ab[s][i]) * SPLIT_UP;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        uint32_t lo, hi;
        take_part(x, lo, hi);
        *reinterpret_cast<uint64_t*>(t.lds + buf * SBUF + p * SPART + sa + i * 32 * SROW) = lo | (uint64_t)hi << 32;
      }
    }
  };
  auto products = [&](int s, int buf) {
    Parts w[2];
    constexpr int AHEAD = MI < 6 ? 1 : 0;  // blocks whose parts are read beforehand: registers
    u32x4_t a[1 + AHEAD][3];
    auto read_a = [&](int i) {
#pragma unroll
      for (int p = 0; p < 3; ++p) a[i & AHEAD][p] = *reinterpret_cast<const u32x4_t*>(t.lds + buf * SBUF + p * SPART + ra + i * 16 * SROW);
    };
    if constexpr (AHEAD) read_a(0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (DIRECT) {
        w[c] = split8(wb[s][2 * c], wb[s][2 * c + 1]);
      } else {
        const char* at = t.lds + buf * TBUF;
        const int rw = own(c) * TLS + lds_rd(r16, kq);
        w[c] = split8(*reinterpret_cast<const u32x4_t*>(at + rw), *reinterpret_cast<const u32x4_t*>(at + (rw ^ 64)));
      }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      if (i + AHEAD < MI) read_a(i + AHEAD);
#pragma unroll
      for (int k = 5; k >= 0; --k) {  // the smallest products first
        constexpr int PW[6] = {0, 0, 1, 1, 0, 2}, PA[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
        for (int c = 0; c < 2; ++c) mma16<uint16_t>(acc[c][i], w[c].p[PW[k]], a[i & AHEAD][PA[k]]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  k_steps<PD>(
      nk,
      [&](int s) {
        load_a(s, s);
        load_w(s, s);
      },
      [&](auto more) {
        store(0, 0);
        if constexpr (more) {
          load_a(0, PD);
          if constexpr (!DIRECT) load_w(0, PD);
        }
      },
      [&](auto s, int kt, auto next, auto more_a, auto more_w) {
        meet();  // buffer kt & 1 is written, the other one read
        if constexpr (next) {
          store((s + 1) % PD, (kt + 1) & 1);
          if constexpr (more_a) {
            load_a((s + 1) % PD, kt + 1 + PD);
            if constexpr (!DIRECT) load_w((s + 1) % PD, kt + 1 + PD);
          }
        }
        products(s, kt & 1);
        if constexpr (DIRECT && more_w) load_w(s, kt + PD);
      });
  if (kb & 127) {  // the rest of K, a multiple of 16 bytes: pieces past the end are zeros
    const int left = kb & 127;
    const u32x4_t zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NA; ++i) ab[0][i] = (tid & 7) * 16 < left ? *reinterpret_cast<const u32x4_t*>(t.ap[i] + nk * 128) : zero;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      wb[0][i] = (DIRECT ? kq * 16 + (i & 1) * 64 : (tid & 7) * 16) < left ? *reinterpret_cast<const u32x4_t*>(t.w + nk * 128 + wp[i]) : zero;
    meet();
    store(0, 0);
    meet();
    products(0, 0);
  }
  // a bit per row of the tile, of all waves together (they hold the rows' other columns)
  if constexpr (!DIRECT) meet();  // (with DIRECT nothing else lies there)
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    bool finite = true;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) finite &= fabsf(acc[c][i][q]) < INFINITY, acc[c][i][q] *= SPLIT_DOWN;
    uint64_t m = __ballot(!finite);
    m |= m >> 32;
    m |= m >> 16;
    if (lane == 0) reinterpret_cast<uint16_t*>(t.lds)[wave * 8 + i] = (uint16_t)m;
  }
  meet();
  uint32_t any = 0, mine = 0;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    uint32_t m = 0;
#pragma unroll
    for (int o = 0; o < 4; ++o) m |= reinterpret_cast<const uint16_t*>(t.lds)[o * 8 + i];
    any |= m;
    mine |= (m >> r16 & 1) << i;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int c = 0; c < (GATED ? 1 : 2); ++c)
      if ((mine >> i & 1) == 0) out(i * 16 + r16, own(c) + kq * 4, acc[c][i], acc[1][i]);
  rows_left = mine;
  return any != 0;
}

// One tile of ``rows`` rows: the body for its size.
template <typename T, bool GATED, typename WRow, typename Out>
__device__ __forceinline__ void run_tile(const MoeTile& t, int rows, WRow wrow, Out out) {
  if constexpr (sizeof(T) == 4) {
    bool left;
    uint32_t which;
    if (rows > 112) left = moe_tile_split<GATED, 8, 2, false>(t, wrow, out, which);
    else if (rows > 96) left = moe_tile_split<GATED, 7, 2, false>(t, wrow, out, which);
    else if (rows > 80) left = moe_tile_split<GATED, 6, 2, false>(t, wrow, out, which);
    else if (rows > 64) left = moe_tile_split<GATED, 5, 2, false>(t, wrow, out, which);
    else if (rows > 48) left = moe_tile_split<GATED, 4, 2, false>(t, wrow, out, which);
    else if (rows > 32) left = moe_tile_split<GATED, 3, 2, false>(t, wrow, out, which);
    else if (rows > 16) left = moe_tile_split<GATED, 2, 3, true>(t, wrow, out, which);
    else left = moe_tile_split<GATED, 1, 3, true>(t, wrow, out, which);
    if (left) {  // rows with infinities and NaNs: as fp32 has them (in the same lanes)
      meet();
      moe_tile_many<T, GATED, 8, 1, 2>(t, wrow, [&](int r, int c, const f32x4_t& g, const f32x4_t& u) {
        if (which >> (r >> 4) & 1) out(r, c, g, u);
      });
    }
    return;
  } else {
    if (rows > 64) return moe_tile_many<T, GATED, 4, 2, 2>(t, wrow, out);
    if (rows > 48) return moe_tile_many<T, GATED, 4, 1, 2>(t, wrow, out);
    if (rows > 32) return moe_tile_many<T, GATED, 3, 1, 2>(t, wrow, out);
    if (rows > 16) return moe_tile_few<T, GATED, 2, 3>(t, wrow, out);
    moe_tile_few<T, GATED, 1, 3>(t, wrow, out);
  }
}

// The work item of a workgroup: expert, tile, block of weight rows; false: none left.
struct Work {
  int e, tile, nb, rows;
};
__device__ __forceinline__ bool find_work(const int* __restrict__ tiles, int NB, Work& w) {
  const int total = tiles[0] * NB, chunk = (total + 7) >> 3;
  const int item = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= chunk || item >= total) return false;
  const int* any = tiles + 1 + 3 * (item / NB);  // a tile of the item's expert
  const int nt = any[2], j = item - any[1] * NB;
  w.nb = j / nt;
  w.tile = any[1] + j % nt;
  w.e = any[0] & 0xffff;
  w.rows = tiles[1 + 3 * w.tile] >> 16;
  return true;
}

// The same, the tiles with the most rows first (order: by_size above). From EVEN tiles on the XCDs take tiles in turn, a tile's
// blocks of weight rows on one of them, whose L2 then holds the tile's rows; an XCD has at most an eighth more of them than the mean.
// With fewer tiles some XCDs would have none or one more: there they take the blocks in turn. fp32, both products with sorting and
// sum, us, tiles by expert / tiles in turn / blocks in turn: 2 experts of 2048 x 5632 and 100 rows 491 / 720 / 491, 4 of 60 rows
// 440 / 535 / 425, 9 of 2048 x 1408 and 60 rows 182 / 238 / 183, 24 of 85 rows 539 / 439 / 395, 64 of 66 rows (71 tiles)
// 1005 / 778 / 763, 128 of 2048 x 768 and 44 rows (128 tiles) 638 / 630 / 638.
constexpr int EVEN = 64;
struct Dealt {
  int rank, nb;  // the tile's place in ``order`` (none from ``total`` on), block of weight rows
};
__host__ __device__ __forceinline__ Dealt deal(int total, int NB, int block) {
  const bool few = total < EVEN;
  const int i = few ? block : block >> 3, j = i / NB;
  return {few ? j : j * 8 + (block & 7), i - j * NB};
}
__device__ __forceinline__ bool find_work_by_size(const int* __restrict__ tiles, const int* __restrict__ order, int NB, Work& w) {
  const Dealt d = deal(tiles[0], NB, blockIdx.x);
  if (d.rank >= tiles[0]) return false;
  w.tile = order[d.rank];
  w.nb = d.nb;
  const int t = tiles[1 + 3 * w.tile];
  w.e = t & 0xffff;
  w.rows = t >> 16;
  return true;
}

}  // namespace moe_tile
