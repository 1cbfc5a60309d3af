// The wide MXFP4 kernel with MXFP8 activations: row blocks of 128 and 160 rows, and which tile a call runs with.
#include "moe_gemm_mxw_kernel.h"

namespace tk {

int32_t gemm_launch_mxw_mx8(const GemmParams& p, MxwTile tile, bool swiglu, bool mx_out, hipStream_t st) {
  if (tile.rows < 128) return gemm_launch_mxw_mx8_low(p, tile, swiglu, mx_out, st);
  return tile.rows == 128 ? launch_mxw<true, 4, 8, 2, 3>(p, swiglu, mx_out, st) : launch_mxw<true, 5, 8, 2, 3>(p, swiglu, mx_out, st);
}

}  // namespace tk
