// The wide MXFP4 kernel with bf16 activations: row blocks of 96 and 160 rows, and which tile a call runs with.
#include "moe_gemm_mxw_kernel.h"

namespace tk {

int32_t gemm_launch_mxw(const GemmParams& p, MxwTile tile, bool swiglu, hipStream_t st) {
  if (tile.rows < 96) return gemm_launch_mxw_low(p, tile, swiglu, st);
  return tile.rows == 96 ? launch_mxw<false, 3, 8, 2, 3>(p, swiglu, false, st) : launch_mxw<false, 5, 8, 2, 2>(p, swiglu, false, st);
}

}  // namespace tk
