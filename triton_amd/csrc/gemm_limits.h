// What a call has to be like for the expert-GEMM kernels that address x through one buffer resource.  Plain C++: the entry point
// (moe_gemm.hip) picks the kernel by it and the host path (host_path.cpp, for both of its callers) the row blocks, so that row
// blocks which only such a kernel has are never chosen for a call that it cannot run.
#pragma once
#include <stdint.h>

namespace tk {

// Slices whose sizes and offsets these kernels keep in registers; other kernels run with more.
constexpr int kDmaSlices = 256;

// Bytes of x for a buffer resource; 0 = x is not one: rows over 2 GiB and more, or rows that overlap (closer together than their
// length: one row expanded to many, sliding windows), whose last ones would reach past rows * stride.
inline uint32_t x_extent(int64_t rows, int64_t stride, int64_t K, int64_t itemsize) {
  const int64_t bytes = rows * stride * itemsize;
  return stride >= K && bytes > 0 && bytes < (int64_t)1 << 31 ? (uint32_t)bytes : 0u;
}

// The memory-to-LDS kernel: x as above, an expert's weights (`w_bytes`) within 2 GiB, the slices in registers.
inline bool dma_runs(uint32_t x_bytes, int64_t n_slices, int64_t w_bytes) {
  return x_bytes != 0 && n_slices <= kDmaSlices && w_bytes < (int64_t)1 << 31;
}

// ... on strided 16-bit weights, whose columns may not overlap either.
inline bool dma_runs_16bit(uint32_t x_bytes, int64_t n_slices, int64_t K, int64_t N, int64_t w_stride_n) {
  return w_stride_n >= K && dma_runs(x_bytes, n_slices, ((N - 1) * w_stride_n + K) * 2);
}

// ... on tiled e4m3 weights (fragments of 32 columns, stages of 256 k, 8 KiB each).
inline bool dma_runs_e4m3(uint32_t x_bytes, int64_t n_slices, int64_t K, int64_t N) {
  return dma_runs(x_bytes, n_slices, (N + 31) / 32 * ((K + 255) / 256) * 8192);
}

// Row blocks (of 64) that the kernel for few rows launches side by side: one a slice at least, and what slices of up to five quarters of
// the mean make, as a random routing does (at 62 rows per slice half of the slices have a second block).
inline int64_t few_row_blocks(int64_t rows, int64_t n_slices) { return n_slices * (rows * 5 / (n_slices * 256) + 1); }

}  // namespace tk
