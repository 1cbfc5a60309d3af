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
  // Tiles of 64 x 64 and 256 of K a stage (the narrow ones of short row blocks) where slices have few rows and those of 128 columns are not two a CU: twice
  // the workgroups read the weights.  Layers, us: 8 experts, top 2, d 2048, d_ff 13312, 28 tokens 154 -> 130; d 1024, d_ff 8192, 128 tokens 87 -> 74; d 2048, d_ff 4096,
  // 200 tokens 74 -> 68; 16 experts, d 1024, d_ff 2560, 108 tokens 52 -> 49; d 1152, d_ff 5120, 406 91.4 -> 90.4.  Up to 52 rows a slice, beyond which slices of over 64,
  // whose tiles stay, are many (62: d 1536, d_ff 2048 48.0 -> 49.2).
  if constexpr (TILE == kDma128 && WK == WK_FP8) {
    const int64_t wide = slices * q.grid_n;
    if (p.M <= slices * 52 && wide * 2 <= dma_grid(p, C::PER_CU, wide * 2)) {
      grid = dma_grid(p, C::PER_CU, wide * 2);
      if (once) return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, true, true>) : launch(moe_gemm_dma_kernel<WK, TILE, false, true, true>);
      return swiglu ? launch(moe_gemm_dma_kernel<WK, TILE, true, true, false>) : launch(moe_gemm_dma_kernel<WK, TILE, false, true, false>);
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
