// bf16 expert GEMM for steps that bring an expert more than a few rows. Two workgroups per CU walk the work items (an expert's tile
// of up to 120 rows, 128 weight rows) as one stream of steps of 64 k each, and the last steps of an item load the first ones of
// the next. Rows and weights go straight to LDS, in rings of their own: the rows, which the XCD's L2 holds, two steps, the
// weights three. Only the pairs of 16-row blocks that hold rows are multiplied (a loop for each number), block b by the
// waves of row b % 2. LDS is what sets the size: 120 rows, so that the two rings and the numbers of the next item's rows are half
// of a CU's. What bounds it: the weights' stream (137 + 71 us for 128 experts of 2048 x 768) while an expert has one tile; with
// more of them the bytes on their way, about 60 KB per CU, against L2's latency under that load.
// Both products with sorting and sum, us, skewed router; in brackets the form before, 128 x 128 tiles through registers to LDS,
// all rows multiplied. 128 experts of 2048 x 768, 8 chosen: 24 rows per expert 247 (253), 40 271 (273), 62 284 (288), 128 346 (353),
// 256 516 (537); 8 of 2048 x 1408: 24 rows 42 (53), 256 rows 66 (79); 8 of 4096 x 8192: 24 rows 340 (336), 96 394 (411), 256 612 (649).
// Over 13 sizes from 100 to 256 rows and four routings each: 32 of 2880 x 2880 7 % faster, 128 of 2048 x 768 2 %, 8 of 4096 x 8192 1 %.
// Slower where an even router gives 112 to 136 rows, so that more experts have a second tile: there up to 14 % with the last, 8 % with
// 128. A koduzen-moe prompt of 2048 takes as long as before (2678), koduzen-hybrid's portions 2529 (2552).
// Taken back: 192 and 240 rows x 256 weight rows with one workgroup per CU are faster where every expert has one tile (128 rows
// each: 168 + 109 against 185 + 117) and lose it to a last round of few items where some have two (207 + 115, 182 + 144
// with that round in halves); 240 x 128 rows 249 + 120.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace moe_ring {

constexpr int NT = 256, ROWS = 120, MA = 4;    // slots of a tile, pairs of blocks of 16 rows
constexpr int NJ = 4, WROWS = 32 * NJ;         // blocks of 16 weight rows per wave, weight rows of an item
constexpr int DA = 2, DW = 3;                  // steps of 64 k that the rings of the activations and the weights hold
constexpr int WIMG = WROWS * 128, AIMG = ROWS * 128, A0 = DW * WIMG;
// behind the rings the next item's row numbers; a tile's last half block, which no row belongs to, is read past its image
constexpr int IDS = A0 + DA * AIMG, LDS = IDS + 2048;
static_assert(A0 + (DA - 1) * AIMG + MA * 4096 <= LDS && LDS <= 80 * 1024, "");  // two workgroups per CU
constexpr uint32_t NOWHERE = 0x80000000u;  // past every buffer's range, whether or not the scalar offset counts in the check

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

// What an item's 128 weight rows are: 128 columns, or 64 gate rows and the matching up rows of a [gate | up] weight.
enum { PLAIN = 0, HALVES = 1 };

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Loads from a buffer straight to LDS (lane l's piece at its size times l). From asm: hipcc counts the LDS reads of a loop only
// when it does not see such a load there.
template <bool WIDE>
__device__ __forceinline__ void dma(i32x4_t rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
  unsigned keep;
  if constexpr (WIDE)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dword %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

__device__ __forceinline__ i32x4_t buffer_of(const void* p, uint32_t bytes) {
  const uint64_t a = (uint64_t)p;
  return i32x4_t{__builtin_amdgcn_readfirstlane((int)a), __builtin_amdgcn_readfirstlane((int)(a >> 32)),
                 __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

__device__ __forceinline__ void mma(f32x4_t& acc, const bf16x8_t& b, const bf16x8_t& a) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pack(float a, float b) {
  const __bf16 x = (__bf16)a, y = (__bf16)b;
  return (uint32_t)__builtin_bit_cast(uint16_t, x) | (uint32_t)__builtin_bit_cast(uint16_t, y) << 16;
}
// rows of 16 lanes: (a0 a1 a2 a3, b0 b1 b2 b3) -> (a0 b0 a2 b2, a1 b1 a3 b3)
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0], b = r[1];
}

template <int N> using Int = std::integral_constant<int, N>;

// tiles, slot_row: moe_tile.h's tables for tiles of ROWS slots. A rows: slot_row / kdiv (kdiv > 0) or the slots themselves.
// N: output columns, a multiple of 8; K: a multiple of 64, at least 256. scale(slot): a row's factor of act; act(g, u, factor): a
// column's value (u: of the gated forms). All byte offsets within A, an expert's weights and slot_row below 2^31.
template <int FORM, typename Scale, typename Act>
__device__ __forceinline__ void run(const uint16_t* __restrict__ A, int64_t a_stride, int kdiv, const int* __restrict__ slot_row,
                                    const int* __restrict__ tiles, const uint16_t* __restrict__ W, int N, int K,
                                    uint16_t* __restrict__ Y, Scale scale, Act act, char* lds) {
  constexpr int H = NJ / 2;
  constexpr int COLS = FORM == PLAIN ? WROWS : WROWS / 2;
  constexpr int STORES = FORM == PLAIN ? NJ / 2 : NJ / 4;  // of a lane for each of its rows
  const int NB = (N + COLS - 1) / COLS, nk = K >> 6;
  const int total = uniform(tiles[0]) * NB, chunk = (total + 7) >> 3, S = gridDim.x >> 3;  // one range of items per XCD
  const int base = (blockIdx.x & 7) * chunk, end = min(total, base + chunk);
  int item = base + (blockIdx.x >> 3);
  if (item >= end) return;

  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wr = w >> 1, wc = w & 1;
  const int wrows = FORM == PLAIN ? N : 2 * N;

  struct Item {
    int tile, rows, col0, mi;
    const uint16_t* w;  // the item's first weight row
    uint32_t bytes;     // from there to the end of the expert's weights
  };
  auto look = [&](int it) {
    const int et = uniform(it / NB);
    const int* any = tiles + 1 + 3 * et;  // a tile of the item's expert
    const int e = uniform(any[0]) & 0xffff, first = uniform(any[1]), nt = uniform(any[2]), j = it - first * NB;
    Item t;
    const int block = uniform(j / nt);
    t.tile = first + j - block * nt;  // the tiles of one block of weight rows side by side
    t.col0 = block * COLS;
    t.rows = uniform(tiles[1 + 3 * t.tile]) >> 16;
    t.mi = (t.rows + 31) >> 5;
    t.w = W + ((int64_t)e * wrows + t.col0) * K;
    t.bytes = (uint32_t)((int64_t)(wrows - t.col0) * K * 2);
    return t;
  };
  // piece j of this wave: rows 8 (n w + j) + (lane >> 3) of an operand of 32 n rows, LDS slot lane & 7 <- chunk
  // (lane & 7) ^ (row / 2 & 7); what is not there is read out of the buffer's range, zeros from nowhere
  uint32_t vw[NJ], va[MA];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int row = 8 * (NJ * w + j) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
    vw[j] = (uint32_t)(FORM == HALVES && row >= WROWS / 2 ? row - WROWS / 2 + N : row) * (uint32_t)(K * 2) + c * 16;
  }
  auto a_row = [&](const Item& t, int j) { return 8 * (t.mi * w + j) + (lane >> 3); };
  auto a_off = [&](const Item& t, int j, int id) {
    const int row = a_row(t, j), c = (lane & 7) ^ ((row >> 1) & 7);
    const int src = kdiv > 0 ? (uint32_t)id / (uint32_t)kdiv : t.tile * ROWS + row;
    return row < t.rows ? (uint32_t)src * (uint32_t)(a_stride * 2) + c * 16 : NOWHERE;
  };
  // A pieces of this wave: the image has no room for the last rows of the last wave
  auto a_pieces = [&](const Item& t) { return min(t.mi, ROWS / 8 - t.mi * w); };
  const i32x4_t ra = buffer_of(A, 0x7fffffffu), ri = buffer_of(slot_row, 0x7fffffffu);
  const uint32_t l0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);

  const int rd0 = fr * 128 + ((fq ^ (fr >> 1)) & 7) * 16, rd1 = rd0 ^ 64;
  const int a_rd = wr * 2048;  // blocks of 16 rows go to the two rows of waves in turn
  auto w_rd = [&](int j) { return (FORM == HALVES ? wc * 8 * NJ + (j % H) * 16 + (j / H) * (WROWS / 2) : wc * 16 * NJ + j * 16) * 128; };

  Item cur = look(item), nxt = cur;
  i32x4_t rw = buffer_of(cur.w, cur.bytes), rn = rw;
#pragma unroll
  for (int j = 0; j < MA; ++j)
    if (j < cur.mi) {
      const int row = a_row(cur, j);
      va[j] = a_off(cur, j, kdiv > 0 && row < cur.rows ? slot_row[cur.tile * ROWS + row] : 0);
    }
  int mi = cur.mi, na = a_pieces(cur);  // of the steps being loaded
  uint32_t wat = 0, aat = A0;           // images of the step being computed
  auto load_a = [&](uint32_t img, uint32_t k, int j) { dma<true>(ra, va[j], k, l0 + img + (mi * w + j) * 1024); };
  auto load_w = [&](uint32_t img, uint32_t k, int j) { dma<true>(rw, vw[j], k, l0 + img + (NJ * w + j) * 1024); };
#pragma unroll
  for (int s = 0; s < DW; ++s) {
    if (s < DA) {
#pragma unroll
      for (int j = 0; j < MA; ++j)
        if (j < na) load_a(A0 + s * AIMG, s * 128, j);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_w(s * WIMG, s * 128, j);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NJ) : "memory");  // the first steps, at least
  __builtin_amdgcn_s_barrier();
  uint32_t ka = (DA - 1) * 128, kw = (DW - 1) * 128;  // bytes into K of the last steps asked for
  bool more = false;
  int behind = 0;  // stores of the last item that surely follow its last loads

  auto run_item = [&](auto MI_) {
    constexpr int MI = decltype(MI_)::value, P = NJ * MI, R = NJ + MI;
    f32x4_t acc[MI][NJ];
    bf16x8_t fa0[MI], fw0[NJ], fa1[MI], fw1[NJ];
    // fragments in the order the products need them: A 0, all of W, A 1 ..
    auto rd = [&](uint32_t wimg, uint32_t aimg, int off, int q, bf16x8_t (&fa)[MI], bf16x8_t (&fw)[NJ]) {
      if (q == 0)
        fa[0] = *reinterpret_cast<const bf16x8_t*>(lds + aimg + a_rd + off);
      else if (q <= NJ)
        fw[q - 1] = *reinterpret_cast<const bf16x8_t*>(lds + wimg + w_rd(q - 1) + off);
      else
        fa[q - NJ] = *reinterpret_cast<const bf16x8_t*>(lds + aimg + a_rd + (q - NJ) * 4096 + off);
    };
    auto reads_before = [](int t) constexpr { return R <= P ? (t < R ? t : R) : (t * R + P - 1) / P; };  // the product t of a half
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < R; ++q) rd(wat, aat, rd0, q, fa0, fw0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // nothing pending on the loop's entry edge
    __builtin_amdgcn_sched_barrier(0);
    // in a form in which no iteration is split off for them
    const int first = K & 63, next_w = uniform(nk - DW), next_a = uniform(nk - DA);
    const int some = uniform(behind >= 4);
#pragma clang loop unroll(disable)
    for (int kt = 0; kt < nk; kt = uniform(kt + 1)) {
#pragma unroll
      for (int t = 0; t < P; ++t) {
        mma(acc[t / NJ][t % NJ], fw0[t % NJ], fa0[t / NJ]);
#pragma unroll
        for (int q = reads_before(t); q < reads_before(t + 1); ++q) rd(wat, aat, rd1, q, fa1, fw1);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the step is in registers; A and W of the next one have landed: in every wave after the barrier. On their way may be the
      // weights of the step after, asked for behind that A, and the last item's stores behind them.
      __builtin_amdgcn_s_waitcnt(0xC07F);
      if (kt == first && some > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NJ + 4) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NJ) : "memory");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t wfree = wat, afree = aat;
      wat = wat == (DW - 1) * WIMG ? 0 : wat + WIMG;
      aat = aat == A0 + (DA - 1) * AIMG ? A0 : aat + AIMG;
      ka += 128, kw += 128;
      if (kt == first && more && kdiv > 0)  // the numbers of the next item's rows
        dma<false>(ri, w * 64 + lane < nxt.rows ? (uint32_t)(nxt.tile * ROWS + w * 64 + lane) * 4 : NOWHERE, 0, l0 + IDS + w * 256);
      if (kt == next_w) {
        rw = rn, kw = 0;
        if (!more) {  // nothing to read
#pragma unroll
          for (int j = 0; j < NJ; ++j) vw[j] = NOWHERE;
        }
      }
      if (kt == next_a) {
        ka = 0;
        mi = nxt.mi;
        na = more ? a_pieces(nxt) : 0;
#pragma unroll
        for (int j = 0; j < MA; ++j)
          if (j < na) va[j] = a_off(nxt, j, kdiv > 0 ? *reinterpret_cast<const int*>(lds + IDS + (a_row(nxt, j) & 255) * 4) : 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < P; ++t) {
        mma(acc[t / NJ][t % NJ], fw1[t % NJ], fa1[t / NJ]);
#pragma unroll
        for (int q = reads_before(t); q < reads_before(t + 1); ++q) rd(wat, aat, rd0, q, fa0, fw0);
#pragma unroll
        for (int q = (t * (MA + NJ) + P - 1) / P; q < ((t + 1) * (MA + NJ) + P - 1) / P; ++q) {
          if (q >= MA) load_w(wfree, kw, q - MA);
          else if (q < na) load_a(afree, ka, q);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // straight from the accumulators (LDS holds the next item's steps): acc[i][j][q] is row 16 (2 i + wr) + fr, weight row
    // 4 fq + q of block j; quarters of the wave exchange blocks so that a lane stores 16 bytes of a row
    behind = cur.col0 + COLS <= N ? (cur.mi - 1) * STORES : 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = 16 * (2 * i + wr) + fr;
      const int64_t slot = (int64_t)cur.tile * ROWS + row;
      uint16_t* y = Y + slot * N + cur.col0;
      const bool live = row < cur.rows;
      const float f = live ? scale(slot) : 1.f;
#pragma unroll
      for (int g = 0; g < STORES; ++g) {
        uint32_t x[2][2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4_t v = acc[i][2 * g + b], u = FORM == HALVES ? acc[i][H + 2 * g + b] : v;
          x[b][0] = pack(act(v[0], u[0], f), act(v[1], u[1], f));
          x[b][1] = pack(act(v[2], u[2], f), act(v[3], u[3], f));
        }
        swap16(x[0][0], x[1][0]);
        swap16(x[0][1], x[1][1]);
        const int n = wc * (FORM == PLAIN ? 16 : 8) * NJ + (2 * g + (fq & 1)) * 16 + (fq >> 1) * 8;
        if (live && cur.col0 + n < N) *reinterpret_cast<u32x4_t*>(y + n) = u32x4_t{x[0][0], x[0][1], x[1][0], x[1][1]};
      }
    }
  };
  while (true) {
    more = item + S < end;
    if (more) {
      nxt = look(item + S);
      rn = buffer_of(nxt.w, nxt.bytes);
    }
    switch (cur.mi) {
      case 1: run_item(Int<1>{}); break;
      case 2: run_item(Int<2>{}); break;
      case 3: run_item(Int<3>{}); break;
      default: run_item(Int<4>{}); break;
    }
    if (!more) break;
    item += S;
    cur = nxt;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // nothing is on its way into LDS that another workgroup may get
}

}  // namespace moe_ring
