// Shared by the ragged-K kernels (ragged_k_gemm.hip: any layout, and aligned operands of short slices; ragged_k_long.hip: aligned operands of long ones).
#pragma once
#include "gemm_common.h"
#include "gemm_limits.h"

namespace tk {

struct RaggedKParams {
  const uint8_t* a;
  int64_t a_stride_m, a_stride_k;  // elements
  const uint8_t* b;
  int64_t b_stride_k, b_stride_n;
  uint8_t* y;
  int64_t y_stride_e, y_stride_m;
  const int32_t* sizes;
  const int32_t* a_offs;
  const int32_t* b_offs;
  int M, N;
  int tiles_m, tiles_n;
  int chunk, n_slices;  // aligned variants: tiles per XCD and turn
  int ahead;            // short slices: how many tiles ahead operands are asked for, 0 = not at all
  int y_dtype;
  uint32_t a_bytes, b_bytes, y_bytes;  // extents for the buffer resources of the aligned variants (y: one slice)
  int a_vec, b_vec;  // the operand's base and strides allow 16-byte loads along its contiguous dimension
};

// Aligned operands (as in tk_ragged_k_gemm), long slices; `tile` = 256 or 128.
int32_t ragged_k_launch_long(const RaggedKParams& p, int dtype, int tile, hipStream_t st);

namespace {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

constexpr int kNonTemporal = 2;  // buffer store: streaming

__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}

template <int DT>
__device__ __forceinline__ f32x16_t mfma_k16(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (DT == TK_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// A fragment of 32 columns by 16 k out of a k-slow stage in LDS: two transposing reads, four k rows (`pitch` bytes each) apart.
__device__ __forceinline__ u32x4_t read_frag_tr(uint32_t at, uint32_t pitch) {
  const uint64_t lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * pitch);
  return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// Rows j * 32 .. + 31 of a wave's 64 columns, 16-bit, into LDS at `sp` as rows of 128 bytes (their 16-byte pieces exchanged by row to spread the
// banks): `c0`, `c1` = the accumulators of columns 0..31 and 32..63 (MFMA with the column side as first operand).
template <int YT>
__device__ __forceinline__ void stage_out_rows(uint8_t* sp, int j, int lane, const f32x16_t& c0, const f32x16_t& c1) {
  const int lr = lane & 31, h = lane >> 5;
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const f32x16_t& c = f ? c1 : c0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint32_t q[4];  // columns 16u + 4h + {01, 23} and 16u + 8 + 4h + {01, 23}
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = YT == TK_BF16 ? pack_bf16x2(c[8 * u + 2 * i], c[8 * u + 2 * i + 1]) : pack_f16x2(c[8 * u + 2 * i], c[8 * u + 2 * i + 1]);
      // after the exchange lanes 0..31 hold columns 16u .. 16u + 7 of their row, lanes 32..63 columns 16u + 8 .. 16u + 15
      const auto s0 = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
      const int r = j * 32 + lr;
      *reinterpret_cast<u32x4_t*>(sp + r * 128 + (((f * 4 + u * 2 + h) ^ (r & 7)) * 16)) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
    }
  }
}
// ... and 16 bytes of row r back, piece pc
__device__ __forceinline__ u32x4_t staged_piece(const uint8_t* sp, int r, int pc) { return *reinterpret_cast<const u32x4_t*>(sp + r * 128 + ((pc ^ (r & 7)) * 16)); }

}  // namespace
}  // namespace tk
