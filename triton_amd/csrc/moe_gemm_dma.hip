// Expert GEMM with both operands staged by memory-to-LDS transfers: square tiles, and which tile a call runs with.
#include "moe_gemm_dma_kernel.h"

namespace tk {
namespace {

template <int WK, int TILE>
int32_t launch_cfg(const GemmParams& p, int grid_m, bool swiglu, hipStream_t st) {
  typedef DmaCfg<TILE> C;
  GemmParams q = p;
  q.grid_n = (int)cdiv(p.N, C::BN);
  const int64_t tiles = (int64_t)grid_m * q.grid_n;
  if (tiles <= 0) return TK_OK;
  if (tiles > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_moe_gemm: grid too large");
  q.total_tiles = (int32_t)tiles;
  unsigned grid = dma_grid(p, C::PER_CU, tiles);
  auto launch = [&](auto kern) -> int32_t {
    if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), C::LDS)) return rc;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(C::NW * 64), C::LDS, st, q);
    return check_launch("moe_gemm_dma_kernel");
  };
  const int64_t slices = p.slice_sizes ? p.n_slices : 1;
  const bool once = reads_once(p.M, slices, C::BM, p.N, p.K * (WK == WK_FP8 ? 1 : 2));
  // Tiles of 64 x 64 and twice the K a stage (the narrow ones that short row blocks have, for all) where those are about one round of two workgroups a CU: the larger
  // ones would be a part of one, and what takes their time is the way of a stage from memory.  Layers, us, 128 x 128 / 64 x 64 (expected tiles of the first and
  // second GEMM where they run): bf16, 8 experts, top 4, d 704, d_ff 1120, 613 tokens 68 / 50 (465 in the second); 8, top 1, 288 and 352, 567 tokens 37 / 26 (141, 64); 16, top 2, 320 and 512,
  // 1146 39 / 31 (219); 8, top 4, 1568 and 256, 699 54 / 45 (381); e4m3, 8, top 2, 2048 and 13312, 28 154 / 130 (256); 1280 and 11904, 234 127 / 105 (226); 1024 and 8192, 128 87 / 74.  One GEMM:
  // bf16, 8 slices of 100, K 512, N 1024 11.4 / 8.5 (264); 16 of 80, K 1024, N 1024 16.2 / 13.7 (448); e4m3, 8 of 80, K 2048, N 2048 16.2 / 14.0 (448), of 200, K 1024, N 2048 13.4 / 12.8.
  // (Half a block a slice more than there are rows for; up to 52 rows a slice, one.)
  if constexpr (TILE == kDma128) {
    const int64_t blocks = p.M <= slices * 52 ? slices : (p.M + slices * 32) / 64, small = blocks * cdiv(p.N, C::SBN);
    if (small <= 512 && small <= dma_grid(p, C::PER_CU, small)) {
      // (a workgroup for every tile that there may be: one with two of them takes twice the time)
      grid = dma_grid(p, C::PER_CU, (cdiv(p.M, 64) + slices) * cdiv(p.N, C::SBN));
      if (once) return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, true, true, true>) : launch(moe_gemm_dma_kernel<WK, TILE, false, true, true, true>);
      return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, true, false, true>) : launch(moe_gemm_dma_kernel<WK, TILE, false, true, false, true>);
    }
  }
  if (once)
    return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, false, true>) : launch(moe_gemm_dma_kernel<WK, TILE, false, false, true>);
  if constexpr (TILE == kDma256) {
    // (the other kernel, half a microsecond faster to start, where all tiles are one round, and its stages are half a percent shorter where they
    // are many: e4m3, K 4096, 31 rounds)
    if (tiles > grid && tiles <= 8 * grid)
      return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, true, false>) : launch(moe_gemm_dma_kernel<WK, TILE, false, true, false>);
  }
  return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, false, false>) : launch(moe_gemm_dma_kernel<WK, TILE, false, false, false>);
}

}  // namespace

int32_t gemm_launch_dma(const GemmParams& p, int wk, DmaTile tile, int grid_m, bool swiglu, hipStream_t st) {
  if (tile.rows == 320) return gemm_launch_dma_tall(p, wk, tile, grid_m, swiglu, st);
  auto launch_16bit = [&](auto wk_c) -> int32_t {
    constexpr int WK = decltype(wk_c)::value;
    return tile.rows == 256 ? launch_cfg<WK, kDma256>(p, grid_m, swiglu, st) : launch_cfg<WK, kDma128>(p, grid_m, swiglu, st);
  };
  switch (wk) {
    case WK_BF16:
      return launch_16bit(template_int<WK_BF16>{});
    case WK_F16:
      return launch_16bit(template_int<WK_F16>{});
    case WK_FP8:
      return tile.rows == 256 ? launch_cfg<WK_FP8, kDma256>(p, grid_m, swiglu, st) : launch_cfg<WK_FP8, kDma128>(p, grid_m, swiglu, st);
  }
  return fail(TK_ERR_INVALID, "tk_moe_gemm: bad weight kind %d", wk);
}

}  // namespace tk
