// bf16 experts of steps that bring each of them few rows (decode): the grouped GEMM bodies of moe_tile.h on this library's
// weight layout - gate and up rows interleaved, [g0, u0, g1, u1, ..] - with SiLU(gate) * up in the first product's epilogue.
// What bounds it is the weights' stream. 512 rows over 128 experts of 2048 x 768, us per product: moe_gemm2 (64 x 128 tiles
// through LDS) 187 + 69, this 138 + 73; both products with sort and sum 257 -> 228, 1600 rows 271 -> 238, 5600 rows 300 -> 259.
#include "llmd_common.h"
#include "moe_tile.h"

using llmd::f2bf;

namespace {

template <bool GATED>
__global__ __launch_bounds__(256, 2) void moe_small_kernel(const uint16_t* __restrict__ A, int64_t a_stride, int topk,
                                                           const int* __restrict__ slot_pair, const int* __restrict__ tiles,
                                                           const uint16_t* __restrict__ Wt, int N, int K,
                                                           uint16_t* __restrict__ Y, int NB) {
  moe_tile::Work wk;
  if (!moe_tile::find_work(tiles, NB, wk)) return;
  __shared__ __attribute__((aligned(128))) char lds[4 * moe_tile::TBUF];
  const int tid = threadIdx.x, col0 = wk.nb * (GATED ? 64 : 128);  // the workgroup's first output column
  const int64_t slot0 = (int64_t)wk.tile * moe_tile::TBM;
  moe_tile::MoeTile t;
  t.K = K, t.lds = lds, t.w = reinterpret_cast<const char*>(Wt + (int64_t)wk.e * (GATED ? 2 * N : N) * K);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // slots past the tile's rows read its last row: their sums are not stored
    const int r = min((tid >> 3) + i * 32, wk.rows - 1);
    const int64_t src = topk > 0 ? slot_pair[slot0 + r] / topk : slot0 + r;
    t.ap[i] = reinterpret_cast<const char*>(A + src * a_stride) + (tid & 7) * 16;
  }
  auto wrow = [&](int j) {  // rows 0 .. 63 gate, 64 .. 127 up; columns past N read the last one
    const int col = min(col0 + (GATED ? j & 63 : j), N - 1);
    return (uint32_t)(GATED ? 2 * col + (j >> 6) : col) * (uint32_t)(K * 2);
  };
  auto out = [&](int r, int c, const moe_tile::f32x4_t& g, const moe_tile::f32x4_t& u) {
    const int n = col0 + c;  // N is a multiple of four
    if (r >= wk.rows || n >= N) return;
    ushort4 b;
    uint16_t* o = &b.x;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = f2bf(GATED ? g[q] / (1.f + __expf(-g[q])) * u[q] : g[q]);
    *reinterpret_cast<ushort4*>(Y + (slot0 + r) * N + n) = b;
  };
  moe_tile::run_tile<uint16_t, GATED>(t, wk.rows, wrow, out);
}

}  // namespace

extern "C" {

// Counters that a sort of n pairs over E experts needs as scratch.
int64_t llmd_moe_sort_scratch(int n, int E) { return moe_sort::many(n, E) ? (int64_t)moe_sort::blocks(n) * E : 0; }

void llmd_moe_group(const int* ids, int n, int E, int* hist, int* slot_pair, int* tiles, int* inv, hipStream_t st) {
  moe_tile::launch_group(ids, n, E, moe_tile::TBM, hist, slot_pair, tiles, inv, nullptr, st);
}

void llmd_moe_small(const void* A, int64_t a_stride, int topk, const int* slot_pair, const int* tiles, int max_tiles,
                    const void* W, int N, int K, void* Y, int gated, hipStream_t st) {
  const int NB = (N + (gated ? 63 : 127)) / (gated ? 64 : 128);
  const dim3 grid((unsigned)(((int64_t)max_tiles * NB + 7) / 8 * 8));
  hipLaunchKernelGGL((gated ? moe_small_kernel<true> : moe_small_kernel<false>), grid, dim3(256), 0, st,
                     (const uint16_t*)A, a_stride, topk, slot_pair, tiles, (const uint16_t*)W, N, K, (uint16_t*)Y, NB);
}

}  // extern "C"
