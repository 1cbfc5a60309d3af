// Expert GEMM, 16-bit operands, about 256 rows per expert: tiles of 320 rows where they make this routing fewer rounds, 256 x 256 ones where not.
//
// Tiles of 320 rows are a fit for slices that are all a little over or under 256 rows, as a random routing makes them; one with favourites has slices of any
// length, and then the larger tiles only divide worse.  The host sees the mean alone, so every workgroup counts both kinds of tiles from the slice
// sizes, all with the same result, and goes on as the kernel for the one that wins.
#include "moe_gemm_dma_kernel.h"

namespace tk {
namespace {

// Which tiles this routing is done with sooner.  320 x 128 tiles are meant for one round (a tile for every workgroup), and a second one costs 45 % more, where
// 256 x 256 tiles stay a part of a round.  320 x 256 tiles cost by full rounds, the started one 0.43 of one (less than one round: by tiles, memory is what
// they share); 256 x 256 ones, the half empty ones among them beside others, 0.73 of such a round for a workgroup's worth of them.
// Measured (rounds in tall tiles / in square ones: us square / tall).  K 2048: 1.00 / 1.25 80 / 84, 1.00 / 1.44 106 / 97, 1.00 / 1.94 140 / 97, 1.06 / 1.97 143 /
// 131, 1.12 / 1.81 130 / 135, 1.31 / 1.44 102 / 144, 2.00 / 2.56 161 / 172, 2.00 / 3.00 177 / 163, 2.06 / 3.00 220 / 229, 2.50 / 3.12 224 / 235, 2.75 / 3.38
// 245 / 242, 2.81 / 3.12 211 / 222, 3.00 / 4.36 300 / 258, 4.50 / 5.75 210 / 213; less than one, K 2880: 0.75 / 0.89 78 / 96, 0.75 / 1.08 110 / 98, 0.84 /
// 0.98 85 / 100, 0.75 / 1.41 123 / 101.  Where slices have more than three square row blocks each, which share their weights, full rounds count on both
// sides, a tall one 5/4 (four live slices of 1150 rows, whole layers: 1.00 / 1.25 173 / 148, of 2048 rows 1.75 / 2.00 209 / 234).  320 x 128: 1.00 / 0.50 56 / 50, 1.06 / 0.56 55 / 74, 1.44 / 0.75 54 / 72.
template <int TILE>
__device__ __forceinline__ bool tall_wins(const GemmParams& p) {
  typedef DmaCfg<TILE> C;
  typedef DmaCfg<kDma256> S;
  int tall = 0, square = 0, live = 0;  // row blocks; slices that have rows
#pragma unroll
  for (int c = 0; c < kSliceRegs; ++c) {
    const int e = c * 64 + (threadIdx.x & 63);
    const int rows = e < p.n_slices ? p.slice_sizes[e] : 0;
    tall += (rows + C::BM - 1) / C::BM, square += (rows + S::BM - 1) / S::BM;
    live += __popcll(__builtin_amdgcn_ballot_w64(rows > 0));
  }
  tall = __builtin_amdgcn_readlane(wave_scan_i32(tall), 63), square = __builtin_amdgcn_readlane(wave_scan_i32(square), 63);
  const bool shared = square > 3 * live;
  tall *= (p.N + C::BN - 1) / C::BN, square *= (p.N + S::BN - 1) / S::BN;
  const int wgs = (int)gridDim.x, full = tall / wgs;
  if constexpr (C::BN < S::BN) return tall <= wgs;
  if (shared) return (tall + wgs - 1) / wgs * 5 <= (square + wgs - 1) / wgs * 4;
  const float rounds = (float)tall / (float)wgs, cost = full == 0 ? rounds : (float)full + (tall > full * wgs ? 0.43f : 0.f);
  return cost < 0.73f * (float)square / (float)wgs;
}

// The kernel's parameters, as the compiler takes it another set of them for each way through a kernel: what both would read alike it reads in front of
// the branch, in scalar registers that neither has to spare (1 to 5 us of 95 for their way out and back).
__device__ __forceinline__ const GemmParams& own_params() {
  auto* q = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(q));
  return *(const GemmParams*)q;
}

// ONCE as in the kernel, for the tall tiles; the square ones, chosen where slices have several row blocks, may cut short ones into narrow tiles.
template <int WK, int TILE, bool SWIGLU, bool ONCE>
__global__ __launch_bounds__(DmaCfg<TILE>::NW * 64, 2) void moe_gemm_dma_tall_kernel(const GemmParams p) {
  static_assert(DmaCfg<TILE>::NW == DmaCfg<kDma256>::NW, "one launch for either");
  if (tall_wins<TILE>(p))
    dma_gemm<WK, TILE, SWIGLU, false, ONCE>(own_params());
  else
    dma_gemm<WK, kDma256, SWIGLU, true, false>(own_params());
}

template <int WK, int TILE>
int32_t launch_tall(const GemmParams& p, int grid_m, bool swiglu, hipStream_t st) {
  typedef DmaCfg<TILE> C;
  constexpr int kLds = C::LDS > DmaCfg<kDma256>::LDS ? C::LDS : DmaCfg<kDma256>::LDS;
  GemmParams q = p;
  q.grid_n = (int)cdiv(p.N, C::BN);
  const int64_t tiles = (int64_t)grid_m * q.grid_n;  // (row blocks of 256, so not fewer than either kind's)
  if (tiles <= 0) return TK_OK;
  if (tiles > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_moe_gemm: grid too large");
  q.total_tiles = (int32_t)tiles;
  auto launch = [&](auto kern) -> int32_t {
    if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), kLds)) return rc;
    hipLaunchKernelGGL(kern, dim3(dma_grid(p, 1, tiles)), dim3(C::NW * 64), kLds, st, q);
    return check_launch("moe_gemm_dma_tall_kernel");
  };
  if (reads_once(p.M, p.n_slices, C::BM, p.N, p.K * 2))
    return swiglu ? launch(moe_gemm_dma_tall_kernel<WK, TILE, true, true>) : launch(moe_gemm_dma_tall_kernel<WK, TILE, false, true>);
  return swiglu ? launch(moe_gemm_dma_tall_kernel<WK, TILE, true, false>) : launch(moe_gemm_dma_tall_kernel<WK, TILE, false, false>);
}

}  // namespace

int32_t gemm_launch_dma_tall(const GemmParams& p, int wk, DmaTile tile, int grid_m, bool swiglu, hipStream_t st) {
  if (wk == WK_BF16) return tile.cols == 256 ? launch_tall<WK_BF16, kDma320>(p, grid_m, swiglu, st) : launch_tall<WK_BF16, kDma320Half>(p, grid_m, swiglu, st);
  if (wk == WK_F16) return tile.cols == 256 ? launch_tall<WK_F16, kDma320>(p, grid_m, swiglu, st) : launch_tall<WK_F16, kDma320Half>(p, grid_m, swiglu, st);
  return fail(TK_ERR_INVALID, "tk_moe_gemm: bad weight kind %d", wk);
}

}  // namespace tk
