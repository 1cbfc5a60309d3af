// The wide MXFP4 kernel with MXFP8 activations and row blocks of 32 and 64 rows.
#include "moe_gemm_mxw_kernel.h"

namespace tk {

int32_t gemm_launch_mxw_mx8_low(const GemmParams& p, MxwTile tile, bool swiglu, bool mx_out, hipStream_t st) {
  return tile.rows == 32 ? launch_mxw<true, 1, 4, 3, 3>(p, swiglu, mx_out, st) : launch_mxw<true, 2, 8, 3, 3>(p, swiglu, mx_out, st);
}

}  // namespace tk
