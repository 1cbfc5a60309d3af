// What the kernels of the decode layer are given (moe_decode_layer.hip and, for small streams of weights, moe_decode_rows.hip).
#pragma once
#include "common.h"
#include "gemm_limits.h"

namespace tk {

struct DecodeParams {
  const uint8_t* x;  // bf16 [T, K1]
  int64_t x_stride;  // elements
  uint32_t x_bytes;  // extent of x (the rows are read through a buffer resource)
  const void* logits;
  int64_t logits_stride;
  int32_t logits_is_bf16;
  int32_t T, E, k, apply_softmax;
  const uint8_t* w1;
  const uint8_t* w1s;
  int64_t w1_stride_e, w1s_stride_e;  // bytes
  const void* b1;
  int64_t b1_stride_e;
  int32_t b1_is_f32;
  const uint8_t* w2;
  const uint8_t* w2s;
  int64_t w2_stride_e, w2s_stride_e;
  const void* b2;
  int64_t b2_stride_e;
  int32_t b2_is_f32;
  int32_t K1, N1, K2, N2;  // K2 = N1 / 2
  int32_t nst1, nst2, nfr1, nfr2;
  float alpha, limit;
  int32_t has_limit;
  uint16_t* h;      // scratch [T*k, K2] bf16, expert-sorted rows
  uint16_t* y;      // scratch [T*k, N2] bf16, flat rows t*k + j
  int32_t* sync;    // [0] finished workgroups, [1] error word, then kDecBlockWords GEMM-1 units done per row block, then [T*nfr2] arrivals
  uint16_t* out;    // [T, N2] bf16
  int64_t out_stride;
  int16_t* indx_out;  // optional [T, k]
  float* vals_out;    // optional [T, k]
  int32_t spin_limit;
};

// The layer row by row in two launches (decode_by_rows); the workspace's y serves as the table between them.
int32_t decode_launch_rows(const DecodeParams& p, hipStream_t st);

}  // namespace tk
