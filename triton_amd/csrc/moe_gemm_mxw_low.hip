// The wide MXFP4 kernel with bf16 activations and row blocks of 32 and 64 rows.
#include "moe_gemm_mxw_kernel.h"

namespace tk {

int32_t gemm_launch_mxw_low(const GemmParams& p, MxwTile tile, bool swiglu, hipStream_t st) {
  if (tile.rows == 32) return launch_mxw<false, 1, 4, 3, 3>(p, swiglu, false, st);
  return tile.cols == 256 ? launch_mxw<false, 2, 4, 2, 2>(p, swiglu, false, st) : launch_mxw<false, 2, 8, 3, 3>(p, swiglu, false, st);
}

}  // namespace tk
