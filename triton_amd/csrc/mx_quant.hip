// MX quantise / dequantise kernels for gfx950 (HBM-bound byte work).
//
// Source layouts handled without a transposed temporary:
//   rows : the quantised axis is the unit-stride one; 4 lanes share a block of 32, each holds 8
//          consecutive elements, the block maximum is a 2-step lane exchange.
//   cols : the quantised axis is strided and the INNER axis is unit-stride (a weight [E, K, N]
//          quantised along K); a lane owns one or two columns and walks 32 rows, so every load of a
//          wave is one contiguous row segment and the 32-element reduction is register-local.
//   tile : the cols case for 16-bit tensors of four columns and more, with an LDS transpose so that the quantised
//          bytes of a column move as full 128-byte lines (mx_down_tile / mx_up_tile); small sources with rows at any
//          address stay with the cols kernel (mx_by_columns).
#include "mx_math.h"
#include "mx_tiles.h"

namespace tk {
namespace {

constexpr int kThreads = 256;

template <int DT>
struct Elem;
template <>
struct Elem<TK_F32> {
  typedef float T;
  static __device__ float load(const T* p) { return *p; }
  static __device__ void store(T* p, float v) { *p = v; }
  static __device__ float max_finite() { return 3.4028234663852886e+38f; }
};
template <>
struct Elem<TK_BF16> {
  typedef uint16_t T;
  static __device__ float load(const T* p) { return bf16_bits_to_f32(*p); }
  static __device__ void store(T* p, float v) { *p = f32_to_bf16_bits(v); }
  static __device__ float max_finite() { return 3.3895313892515355e+38f; }
};
template <>
struct Elem<TK_F16> {
  typedef uint16_t T;
  static __device__ float load(const T* p) { return f16_bits_to_f32(*p); }
  static __device__ void store(T* p, float v) { *p = f32_to_f16_bits(v); }
  static __device__ float max_finite() { return 65504.0f; }
};

// Index of the output line (run of one (outer, inner) coordinate along the quantised axis).  The inner
// extent is mid x last with `last` fastest in the source; outputs order lines (outer, last, mid), which
// is the order `x.transpose(axis, -1)` gives them.
__device__ inline int64_t line_of(int64_t o, int64_t col, int64_t inner, int64_t inner_last) {
  if (inner_last == inner) return o * inner + col;
  const int64_t m = col / inner_last;
  const int64_t l = col - m * inner_last;
  return (o * inner_last + l) * (inner / inner_last) + m;
}

typedef __attribute__((ext_vector_type(2))) unsigned short u16x2_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a), __builtin_bit_cast(u16x2_t, b)));
}
// two 16-bit floats (low half first) / scale -> two e2m1 codes in byte `SEL` of `old` (first value in the low nibble)
template <int SRC>
__device__ __forceinline__ uint32_t cvt_pk_fp4(uint32_t old, uint32_t pair, float scale, int sel) {
  if constexpr (SRC == TK_BF16) {
    const bf16x2_t v = __builtin_bit_cast(bf16x2_t, pair);
    return sel == 0   ? __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(old, v, scale, 0)
           : sel == 1 ? __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(old, v, scale, 1)
           : sel == 2 ? __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(old, v, scale, 2)
                      : __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(old, v, scale, 3);
  } else {
    const f16x2_t v = __builtin_bit_cast(f16x2_t, pair);
    return sel == 0   ? __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(old, v, scale, 0)
           : sel == 1 ? __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(old, v, scale, 1)
           : sel == 2 ? __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(old, v, scale, 2)
                      : __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(old, v, scale, 3);
  }
}

// byte pair `SEL` of `w` (two e2m1 codes, low nibble first) * scale -> two 16-bit floats (first value in the low half)
template <int DST>
__device__ __forceinline__ uint32_t cvt_pk_from_fp4(uint32_t w, float scale, int sel) {
  if constexpr (DST == TK_BF16) {
    const bf16x2_t r = sel == 0   ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 0)
                       : sel == 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 1)
                       : sel == 2 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 2)
                                  : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 3);
    return __builtin_bit_cast(uint32_t, r);
  } else {
    const f16x2_t r = sel == 0   ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 0)
                      : sel == 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 1)
                      : sel == 2 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 2)
                                 : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, scale, 3);
    return __builtin_bit_cast(uint32_t, r);
  }
}

// The hardware's 8-bit float conversions give the bytes of the bit algorithms in mx_math.h: compared on the GPU over every 16-bit pattern under every
// scale (down) and every code under every scale (up), they differ in overflow (a value past the largest finite one gives NaN; here it saturates), in the
// sign and payload of NaN, and where a product with the scale leaves the target type's range.  Calls clamp, or exclude, those.
// Two fp32 -> two bytes (first in the low one), saturating; NaN becomes 0x7F with its sign.
template <int KIND>
__device__ __forceinline__ uint32_t quant_pair(float q0, float q1) {
  const float mq = KIND == TK_E4M3 ? 448.0f : 57344.0f;
  const uint32_t w = (uint32_t)(KIND == TK_E4M3 ? __builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp(q0, mq), mx_clamp(q1, mq), 0, false)
                                                : __builtin_amdgcn_cvt_pk_bf8_f32(mx_clamp(q0, mq), mx_clamp(q1, mq), 0, false));
  const uint32_t lo = q0 != q0 ? ((hd_f32_bits(q0) >> 24) & 0x80u) | 0x7Fu : w & 0xFFu;
  const uint32_t hi = q1 != q1 ? ((hd_f32_bits(q1) >> 16) & 0x8000u) | 0x7F00u : w & 0xFF00u;
  return lo | hi;
}

// two 16-bit floats (low half first) / scale -> two bytes in half `sel` of `old`; the quotients must be finite and within the format's range
template <int SRC, int KIND>
__device__ __forceinline__ uint32_t cvt_pk_8(uint32_t old, uint32_t pair, float scale, int sel) {
  typedef __attribute__((ext_vector_type(2))) short s16x2_t;
  const s16x2_t o = __builtin_bit_cast(s16x2_t, old);
  s16x2_t r;
  if constexpr (SRC == TK_BF16) {
    const bf16x2_t v = __builtin_bit_cast(bf16x2_t, pair);
    if constexpr (KIND == TK_E4M3)
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(o, v, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(o, v, scale, true);
    else
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf8_bf16(o, v, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_bf8_bf16(o, v, scale, true);
  } else {
    const f16x2_t v = __builtin_bit_cast(f16x2_t, pair);
    if constexpr (KIND == TK_E4M3)
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(o, v, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(o, v, scale, true);
    else
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf8_f16(o, v, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_bf8_f16(o, v, scale, true);
  }
  return __builtin_bit_cast(uint32_t, r);
}

// half `sel` of `w` (two bytes, low one first) * scale -> two 16-bit floats; no NaN or infinity among the codes and a scale of `up_scale_ok`
template <int KIND, int DST>
__device__ __forceinline__ uint32_t cvt_pk_from_8(uint32_t w, float scale, int sel) {
  if constexpr (DST == TK_BF16) {
    bf16x2_t r;
    if constexpr (KIND == TK_E4M3)
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, true);
    else
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, scale, true);
    return __builtin_bit_cast(uint32_t, r);
  } else {
    f16x2_t r;
    if constexpr (KIND == TK_E4M3)
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, scale, true);
    else
      r = sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, scale, false) : __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, scale, true);
    return __builtin_bit_cast(uint32_t, r);
  }
}

// Scales (e8m0 bytes) under which the conversion above equals dequantising in fp32, clamping to the target's range and rounding: no finite code leaves
// that range.  (e2m1: see mx_up_tile.)
template <int KIND, int DST>
__device__ __forceinline__ bool up_scale_ok(uint32_t sb) {
  if (KIND == TK_E2M1) return DST == TK_BF16 ? (sb >= 8 && sb <= 248) : (sb >= 114 && sb <= 139);
  const uint32_t top = KIND == TK_E4M3 ? (DST == TK_BF16 ? 246u : 134u) : (DST == TK_BF16 ? 239u : 127u);
  return sb >= 1 && sb <= top;
}
// scale bits under which the packed conversions of finite 16-bit elements need no clamp and lose nothing.  (e2m1 saturates by itself; extreme scales, where
// subnormal elements could matter, are left out.  fp8: the scale rounded up, so that max / scale is within the format's range.)
template <int KIND>
__device__ __forceinline__ bool down_scale_ok(uint32_t sb, int rounding) {
  if (KIND == TK_E2M1) return sb >= (16u << 23) && sb <= (250u << 23);
  return rounding == TK_MX_ROUND_UP && sb >= (1u << 23) && sb <= (254u << 23);
}
// nonzero where one of a word's four codes is NaN (e4m3) or NaN or an infinity (e5m2)
template <int KIND>
__device__ __forceinline__ uint32_t special_codes(uint32_t w) {
  return ((w & 0x7F7F7F7Fu) + (KIND == TK_E4M3 ? 0x01010101u : 0x04040404u)) & 0x80808080u;
}

template <int KIND>
__device__ inline float elem_f32(uint32_t b) {
  if (KIND == TK_E4M3) return e4m3_to_f32(b);
  return e5m2_to_f32(b);
}

// ---------------------------------------------------------------------------------------------
// downcast, quantised axis contiguous: src [rows, L] with row stride `ld`
// ---------------------------------------------------------------------------------------------
// One lane takes eight elements (16 bytes of a 16-bit tensor in one load), the four lanes of a block share its maximum.  16-bit sources whose block is finite
// (and, for fp8, whose scale is rounded up, so that no quotient passes the largest finite code) go through the packed conversions, one instruction for
// two elements; everything else takes the fp32 path.  A row index is a division, in 32 bits where the indices fit.
template <int SRC, int KIND>
__global__ __launch_bounds__(kThreads) void mx_down_rows(const typename Elem<SRC>::T* __restrict__ src, int64_t ld,
                                                         int64_t rows, int64_t L, uint8_t* __restrict__ out_vals,
                                                         uint8_t* __restrict__ out_scales, int rounding) {
  typedef typename Elem<SRC>::T T;
  const int64_t groups_per_row = L / 8;
  const int64_t total = rows * groups_per_row;
  const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (gid >= total) return;  // total % 4 == 0, so a quad of lanes is either fully in or fully out
  const int64_t row = total <= 0xFFFFFFFFll ? (int64_t)((uint32_t)gid / (uint32_t)groups_per_row) : gid / groups_per_row;
  const int64_t g = gid - row * groups_per_row;
  T e[8];
  __builtin_memcpy(e, src + row * ld + g * 8, sizeof(e));
  uint8_t* const dst = out_vals + row * (KIND == TK_E2M1 ? L / 2 : L) + g * (KIND == TK_E2M1 ? 4 : 8);
  uint8_t* const sdst = out_scales + row * (L / 32) + (g >> 2);
  float m = 0.0f;
  if constexpr (sizeof(T) == 2) {
    uint32_t w[4], mx = 0;
    __builtin_memcpy(w, e, 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) mx = pk_max_u16(mx, w[i] & 0x7FFF7FFFu);
    mx = pk_max_u16(mx, (uint32_t)__shfl_xor((int)mx, 1));
    mx = pk_max_u16(mx, (uint32_t)__shfl_xor((int)mx, 2));
    const uint32_t m16 = mx >> 16 > (mx & 0xFFFFu) ? mx >> 16 : mx & 0xFFFFu;
    const float mf = SRC == TK_BF16 ? hd_bits_f32(m16 << 16) : f16_bits_to_f32((uint16_t)m16);
    const uint32_t sb = mx_scale_bits(mf, KIND, rounding);
    const bool finite = SRC == TK_BF16 ? m16 < 0x7F80u : m16 < 0x7C00u;
    if (finite && down_scale_ok<KIND>(sb, rounding)) {
      const float scale = hd_bits_f32(sb);
      if constexpr (KIND == TK_E2M1) {
        uint32_t o = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) o = cvt_pk_fp4<SRC>(o, w[i], scale, i);
        *reinterpret_cast<uint32_t*>(dst) = o;
      } else {
        uint32_t o[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i >> 1] = cvt_pk_8<SRC, KIND>(o[i >> 1], w[i], scale, i & 1);
        *reinterpret_cast<uint2*>(dst) = make_uint2(o[0], o[1]);
      }
      if ((g & 3) == 0) *sdst = (uint8_t)(sb >> 23);
      return;  // all four lanes of a block come to the same answer
    }
  }
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[i] = Elem<SRC>::load(e + i);
    m = fmaxf(m, fabsf(v[i]));
  }
  m = fmaxf(m, __shfl_xor(m, 1));
  m = fmaxf(m, __shfl_xor(m, 2));
  const uint32_t sbits = mx_scale_bits(m, KIND, rounding);
  const float inv = mx_inv_scale(sbits);
  if (KIND == TK_E2M1) {
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) packed |= e2m1_code(v[i] * inv) << (4 * i);
    *reinterpret_cast<uint32_t*>(dst) = packed;
  } else {
    uint32_t o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) o[h] = quant_pair<KIND>(v[4 * h] * inv, v[4 * h + 1] * inv) | quant_pair<KIND>(v[4 * h + 2] * inv, v[4 * h + 3] * inv) << 16;
    *reinterpret_cast<uint2*>(dst) = make_uint2(o[0], o[1]);
  }
  if ((g & 3) == 0) *sdst = (uint8_t)(sbits >> 23);
}

// ---------------------------------------------------------------------------------------------
// downcast, inner axis contiguous: src [outer, L, inner], stride_inner == 1
// tile = 4 blocks of 32 rows x (64*CPT) columns per 256-thread workgroup; wave w owns block w
// ---------------------------------------------------------------------------------------------
template <int SRC, int KIND, int CPT>
__global__ __launch_bounds__(kThreads) void mx_down_cols(const typename Elem<SRC>::T* __restrict__ src,
                                                         int64_t stride_outer, int64_t stride_axis, int64_t L,
                                                         int64_t inner, int64_t inner_last, int64_t col_tiles,
                                                         int64_t blk_tiles, uint8_t* __restrict__ out_vals,
                                                         uint8_t* __restrict__ out_scales, int rounding) {
  typedef typename Elem<SRC>::T T;
  int64_t bid = blockIdx.x;
  const int64_t ct = bid % col_tiles;
  bid /= col_tiles;
  const int64_t bt = bid % blk_tiles;
  const int64_t o = bid / blk_tiles;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t blk = bt * 4 + wave;
  const int64_t col = (ct * 64 + lane) * CPT;
  if (blk >= L / 32 || col >= inner) return;
  const T* p = src + o * stride_outer + blk * 32 * stride_axis + col;
  float v[32][CPT];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    if (CPT == 2) {
      if (sizeof(T) == 2) {
        uint32_t w = *reinterpret_cast<const uint32_t*>(p + i * stride_axis);
        uint16_t a = (uint16_t)(w & 0xFFFFu), b = (uint16_t)(w >> 16);
        v[i][0] = Elem<SRC>::load(reinterpret_cast<const T*>(&a));
        v[i][CPT - 1] = Elem<SRC>::load(reinterpret_cast<const T*>(&b));
      } else {
        float2 w = *reinterpret_cast<const float2*>(p + i * stride_axis);
        v[i][0] = w.x;
        v[i][CPT - 1] = w.y;
      }
    } else {
      v[i][0] = Elem<SRC>::load(p + i * stride_axis);
    }
  }
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) m = fmaxf(m, fabsf(v[i][c]));
    const uint32_t sbits = mx_scale_bits(m, KIND, rounding);
    const float inv = mx_inv_scale(sbits);
    const int64_t line = line_of(o, col + c, inner, inner_last);
    if (KIND == TK_E2M1) {
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 32; ++i) w[i >> 3] |= e2m1_code(v[i][c] * inv) << (4 * (i & 7));
      *reinterpret_cast<uint4*>(out_vals + line * (L / 2) + blk * 16) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
      uint32_t w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        w[i] = quant_pair<KIND>(v[4 * i][c] * inv, v[4 * i + 1][c] * inv) | quant_pair<KIND>(v[4 * i + 2][c] * inv, v[4 * i + 3][c] * inv) << 16;
      uint4* dst = reinterpret_cast<uint4*>(out_vals + line * L + blk * 32);
      dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
      dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
    }
    out_scales[line * (L / 32) + blk] = (uint8_t)(sbits >> 23);
  }
}

// ---------------------------------------------------------------------------------------------
// upcast, quantised axis contiguous in the output: out [rows, L] with row stride `ld`
// ---------------------------------------------------------------------------------------------
template <int KIND, int DST>
__global__ __launch_bounds__(kThreads) void mx_up_rows(const uint8_t* __restrict__ vals,
                                                       const uint8_t* __restrict__ scales, int64_t rows, int64_t L,
                                                       typename Elem<DST>::T* __restrict__ out, int64_t ld) {
  const int64_t groups_per_row = L / 8;
  const int64_t total = rows * groups_per_row;
  const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (gid >= total) return;
  const int64_t row = gid / groups_per_row;
  const int64_t g = gid - row * groups_per_row;
  const uint32_t sb = scales[row * (L / 32) + (g >> 2)];
  const float mf = Elem<DST>::max_finite();
  float v[8];
  if (KIND == TK_E2M1) {
    const uint32_t packed = *reinterpret_cast<const uint32_t*>(vals + row * (L / 2) + g * 4);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = mx_dequant(bf16_bits_to_f32((uint16_t)e2m1_to_bf16_bits((packed >> (4 * i)) & 0xFu)), sb, mf, false);
  } else {
    const uint2 w = *reinterpret_cast<const uint2*>(vals + row * L + g * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = mx_dequant(elem_f32<KIND>((w.x >> (8 * i)) & 0xFFu), sb, mf, KIND == TK_E5M2);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[4 + i] = mx_dequant(elem_f32<KIND>((w.y >> (8 * i)) & 0xFFu), sb, mf, KIND == TK_E5M2);
  }
  typename Elem<DST>::T* q = out + row * ld + g * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i) Elem<DST>::store(q + i, v[i]);
}

// ---------------------------------------------------------------------------------------------
// upcast, inner axis contiguous in the output: out [outer, L, inner], ostride_inner == 1
// ---------------------------------------------------------------------------------------------
template <int KIND, int DST, int CPT>
__global__ __launch_bounds__(kThreads) void mx_up_cols(const uint8_t* __restrict__ vals,
                                                       const uint8_t* __restrict__ scales, int64_t L, int64_t inner,
                                                       int64_t inner_last, int64_t col_tiles, int64_t blk_tiles,
                                                       typename Elem<DST>::T* __restrict__ out,
                                                       int64_t ostride_outer, int64_t ostride_axis) {
  typedef typename Elem<DST>::T T;
  int64_t bid = blockIdx.x;
  const int64_t ct = bid % col_tiles;
  bid /= col_tiles;
  const int64_t bt = bid % blk_tiles;
  const int64_t o = bid / blk_tiles;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t blk = bt * 4 + wave;
  const int64_t col = (ct * 64 + lane) * CPT;
  if (blk >= L / 32 || col >= inner) return;
  const float mf = Elem<DST>::max_finite();
  float v[32][CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int64_t line = line_of(o, col + c, inner, inner_last);
    const uint32_t sb = scales[line * (L / 32) + blk];
    if (KIND == TK_E2M1) {
      const uint4 w4 = *reinterpret_cast<const uint4*>(vals + line * (L / 2) + blk * 16);
      const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
      for (int i = 0; i < 32; ++i)
        v[i][c] = mx_dequant(bf16_bits_to_f32((uint16_t)e2m1_to_bf16_bits((w[i >> 3] >> (4 * (i & 7))) & 0xFu)), sb,
                             mf, false);
    } else {
      const uint4* src = reinterpret_cast<const uint4*>(vals + line * L + blk * 32);
      const uint4 a = src[0], b = src[1];
      const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 32; ++i)
        v[i][c] = mx_dequant(elem_f32<KIND>((w[i >> 2] >> (8 * (i & 3))) & 0xFFu), sb, mf, KIND == TK_E5M2);
    }
  }
  T* q = out + o * ostride_outer + blk * 32 * ostride_axis + col;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    if (CPT == 2 && sizeof(T) == 2) {
      uint16_t a, b;
      Elem<DST>::store(reinterpret_cast<T*>(&a), v[i][0]);
      Elem<DST>::store(reinterpret_cast<T*>(&b), v[i][CPT - 1]);
      *reinterpret_cast<uint32_t*>(q + i * ostride_axis) = (uint32_t)a | ((uint32_t)b << 16);
    } else if (CPT == 2) {
      *reinterpret_cast<float2*>(q + i * ostride_axis) = make_float2(v[i][0], v[i][CPT - 1]);
    } else {
      Elem<DST>::store(q + i * ostride_axis, v[i][0]);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// 16-bit sources / destinations with the inner axis contiguous, through an LDS transpose.
// A workgroup takes 256 columns x NB blocks of 32 rows, NB chosen so that the NB blocks of one column are
// 128 output bytes (8 blocks of e2m1, 4 of fp8): the quantised bytes of a column are then moved as one full
// 128-byte line (8 lanes x 16 bytes) instead of 16- or 32-byte pieces of 64 different lines per instruction,
// and a lane walks its rows with 8-byte accesses (4 columns), so a wave covers 512 contiguous bytes per row.
// ---------------------------------------------------------------------------------------------
constexpr int kTileCols = kMxTileCols;
constexpr int kTilePitch = 128 + 16;  // LDS bytes per column
// LDS row of tile column c: a lane's four adjacent columns are spread 65 rows apart, so the 16-byte accesses of
// consecutive lanes (columns c, c + 4, ...) fall 144 bytes apart and take different banks
constexpr int kTileRows = 64 + 65 * 3;
__device__ __forceinline__ int tile_row(int c) { return (c >> 2) + 65 * (c & 3); }
// First column of tile `ct`, and the first of a lane's four columns inside it.  Where the number of columns is no multiple of four (it is at least four),
// the last lane moves back to end with the last column and does up to three columns again that its neighbour does, with the same result.  Rows then start
// at any even address: the memory takes 8 bytes a lane at any alignment, and the 512 bytes of a wave's row touch one line more.  (6 x 1632 x 1093 to e4m3 and
// back, a column per lane and 16 or 32 bytes of a line per store: 15.3 + 15.2 us; this way 9.6 + 10.4.)
__device__ __forceinline__ int64_t tile_col0(int64_t ct, int64_t inner) { return ct * kTileCols < inner - 4 ? ct * kTileCols : inner - 4; }
__device__ __forceinline__ int tile_cols_of(int lane, int64_t col0, int64_t inner) {
  const int64_t last = inner - 4 - col0;
  return lane * 4 < last ? lane * 4 : (int)last;
}
// 8 bytes at any even address
typedef __attribute__((ext_vector_type(2), aligned(2))) uint32_t u32x2_any_t;

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Tiles are renumbered so that consecutive
// tiles run on ONE XCD at about the same time, and the tiles of one column range are numbered consecutively along
// the quantised axis: a column's quantised bytes (1440 per 2880 values of e2m1) are not a multiple of the 128-byte
// line, so neighbouring tiles share the lines at their seams and the 64-byte pieces of the scale rows; in one L2
// those are fetched (or written back) once, in two L2s twice.
__device__ __forceinline__ int64_t tile_order(int64_t pid, int64_t total) {
  const int64_t per = total / 8, extra = total % 8;
  const int64_t grp = pid % 8, local = pid / 8;
  return grp * per + (grp < extra ? grp : extra) + local;
}

template <int KIND>
struct TileGeom {
  static constexpr int BB = KIND == TK_E2M1 ? 16 : 32;  // value bytes per block and column
  static constexpr int NB = mx_tile_blocks(KIND == TK_E2M1), SMALL = kMxSmallBlocks;  // blocks per tile
  static_assert(NB * BB == 128, "a column of a tile is a whole line");
};

// The tile's value bytes and scales from LDS to global memory.  Scales: a column's NB bytes are contiguous in both places, so one thread moves them in one piece
// (4 or 8 bytes at any alignment) unless the tile hangs over the end of the axis; single-byte accesses cost an instruction and a memory transaction each.
template <int KIND, int NB>
__device__ __forceinline__ void tile_store(const uint8_t* vals_s, const uint8_t* sc_s, uint8_t* gvals, uint8_t* gscales, int64_t o, int64_t col0,
                                           int64_t blk0, int64_t L, int64_t inner, int64_t inner_last) {
  constexpr int BB = TileGeom<KIND>::BB, PIECES = NB * BB / 16;  // (of a column)
  const int64_t nblk = L / 32;
  const int64_t line_bytes = KIND == TK_E2M1 ? L / 2 : L;
#pragma unroll
  for (int it = 0; it < PIECES; ++it) {
    const int q = it * kThreads + threadIdx.x;
    const int col = q / PIECES, piece = q % PIECES;
    const int64_t blk = blk0 + piece * 16 / BB;
    if (col0 + col < inner && blk < nblk) {
      const int64_t line = line_of(o, col0 + col, inner, inner_last);
      *reinterpret_cast<uint4*>(gvals + line * line_bytes + blk0 * BB + piece * 16) = *reinterpret_cast<const uint4*>(vals_s + tile_row(col) * kTilePitch + piece * 16);
    }
  }
  static_assert(kTileCols == kThreads, "one column per thread");
  const int col = threadIdx.x;
  if (col0 + col < inner && blk0 < nblk) {
    uint8_t* g = gscales + line_of(o, col0 + col, inner, inner_last) * nblk + blk0;
    const uint8_t* l = sc_s + col * NB;
    if (blk0 + NB <= nblk)
      __builtin_memcpy(g, l, NB);
    else
      for (int b = 0; blk0 + b < nblk; ++b) g[b] = l[b];
  }
}

// ... and from global memory to LDS.  TOGETHER: everything is requested before any of it is written to LDS, without a condition around a load, whose end would wait for it; a
// thread past the last column or block fetches that one again, for a place that nobody reads.  One piece after the other a tile is up to nine round trips, which is what a launch
// of few tiles takes; with many tiles a CU others run meanwhile, and fewer requests at a time serve the memory better (mx_tiles).
template <int KIND, int NB, bool TOGETHER>
__device__ __forceinline__ void tile_fetch(uint8_t* vals_s, uint8_t* sc_s, const uint8_t* gvals, const uint8_t* gscales, int64_t o, int64_t col0,
                                           int64_t blk0, int64_t L, int64_t inner, int64_t inner_last) {
  constexpr int BB = TileGeom<KIND>::BB, PIECES = NB * BB / 16;
  const int64_t nblk = L / 32;
  const int64_t line_bytes = KIND == TK_E2M1 ? L / 2 : L;
  if constexpr (!TOGETHER) {
#pragma unroll
    for (int it = 0; it < PIECES; ++it) {
      const int q = it * kThreads + threadIdx.x;
      const int col = q / PIECES, piece = q % PIECES;
      if (col0 + col < inner && blk0 + piece * 16 / BB < nblk)
        *reinterpret_cast<uint4*>(vals_s + tile_row(col) * kTilePitch + piece * 16) =
            *reinterpret_cast<const uint4*>(gvals + line_of(o, col0 + col, inner, inner_last) * line_bytes + blk0 * BB + piece * 16);
    }
    const int col = threadIdx.x;
    if (col0 + col < inner) {
      const uint8_t* g = gscales + line_of(o, col0 + col, inner, inner_last) * nblk + blk0;
      uint8_t* l = sc_s + col * NB;
      if (blk0 + NB <= nblk)
        __builtin_memcpy(l, g, NB);
      else
        for (int b = 0; blk0 + b < nblk; ++b) l[b] = g[b];
    }
    return;
  }
  auto line = [&](int col) __attribute__((always_inline)) { return line_of(o, col0 + col < inner ? col0 + col : inner - 1, inner, inner_last); };
  uint8_t sc[NB];
  const uint8_t* gs = gscales + line(threadIdx.x) * nblk;
  if (blk0 + NB <= nblk) {
    __builtin_memcpy(sc, gs + blk0, NB);
  } else {
#pragma unroll
    for (int b = 0; b < NB; ++b) sc[b] = gs[blk0 + b < nblk ? blk0 + b : nblk - 1];
  }
  uint4 v[PIECES];
#pragma unroll
  for (int it = 0; it < PIECES; ++it) {
    const int q = it * kThreads + threadIdx.x, byte = q % PIECES * 16;
    const int64_t blk = blk0 + byte / BB;
    v[it] = *reinterpret_cast<const uint4*>(gvals + line(q / PIECES) * line_bytes + (blk < nblk ? blk : nblk - 1) * BB + byte % BB);
  }
  __builtin_memcpy(sc_s + threadIdx.x * NB, sc, NB);
#pragma unroll
  for (int it = 0; it < PIECES; ++it) {
    const int q = it * kThreads + threadIdx.x;
    *reinterpret_cast<uint4*>(vals_s + tile_row(q / PIECES) * kTilePitch + q % PIECES * 16) = v[it];
  }
}

// Quantises the lane's 32 rows x 4 columns of block `b` (raw[i] = row i, two 16-bit elements per dword) into the
// tile's LDS staging arrays.
template <int SRC, int KIND, int NB>
__device__ __forceinline__ void quantise_block_to_lds(const uint2 (&raw)[32], uint8_t* vals_s, uint8_t* sc_s, int c4, int b, int rounding) {
  constexpr int BB = TileGeom<KIND>::BB;
  // The block maxima come from the 16-bit patterns themselves (|x| orders like its bits without the sign, two elements per instruction) and the
  // hardware converts two 16-bit floats to two codes while dividing by the power-of-two scale (round to nearest even, exact), so a pair of rows costs
  // one byte permute and one conversion.  A lane with a block that holds an infinity or a NaN, or whose scale is outside `down_scale_ok`, takes the fp32
  // path below, as a loop over its columns: the bit algorithms of fp8, unrolled over the 128 elements, were 25 KB of instructions, and fetching those was
  // most of the time of a small tensor (2 x 64 x 528 e5m2: 20 us a launch, 4.6 now; 32 x 2880 x 5760 e4m3: 395 us, 300 with the hint below).
  uint32_t max01 = 0, max23 = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    max01 = pk_max_u16(max01, raw[i].x & 0x7FFF7FFFu);
    max23 = pk_max_u16(max23, raw[i].y & 0x7FFF7FFFu);
  }
  uint32_t sb[4];
  bool fast = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t mx = c < 2 ? max01 : max23;
    const uint32_t m16 = (c & 1) ? (mx >> 16) : (mx & 0xFFFFu);
    sb[c] = mx_scale_bits(SRC == TK_BF16 ? hd_bits_f32(m16 << 16) : f16_bits_to_f32((uint16_t)m16), KIND, rounding);
    fast = fast && (SRC == TK_BF16 ? m16 < 0x7F80u : m16 < 0x7C00u) && down_scale_ok<KIND>(sb[c], rounding);
  }
  if (fast) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint4* dst = reinterpret_cast<uint4*>(vals_s + tile_row(c4 + c) * kTilePitch + b * BB);
      const float scale = hd_bits_f32(sb[c]);
      uint32_t w[BB / 4];
#pragma unroll
      for (int i = 0; i < BB / 4; ++i) w[i] = 0;
#pragma unroll
      for (int i = 0; i < 32; i += 2) {
        const uint32_t lo = c < 2 ? raw[i].x : raw[i].y, hi = c < 2 ? raw[i + 1].x : raw[i + 1].y;
        const uint32_t pair = __builtin_amdgcn_perm(hi, lo, (c & 1) ? 0x07060302u : 0x05040100u);  // (row i, row i+1) of column c
        if constexpr (KIND == TK_E2M1)
          w[i >> 3] = cvt_pk_fp4<SRC>(w[i >> 3], pair, scale, (i >> 1) & 3);
        else
          w[i >> 2] = cvt_pk_8<SRC, KIND>(w[i >> 2], pair, scale, (i >> 1) & 1);
      }
#pragma unroll
      for (int i = 0; i < BB / 16; ++i) dst[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
      sc_s[(c4 + c) * NB + b] = (uint8_t)(sb[c] >> 23);
    }
    return;
  }
#pragma unroll 1
  for (int c = 0; c < 4; ++c) {
    auto elem = [&](int i) __attribute__((always_inline)) {
      const uint16_t e = (uint16_t)((c < 2 ? raw[i].x : raw[i].y) >> (16 * (c & 1)));
      return Elem<SRC>::load(&e);
    };
    uint4* dst = reinterpret_cast<uint4*>(vals_s + tile_row(c4 + c) * kTilePitch + b * BB);
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) m = fmaxf(m, fabsf(elem(i)));
    const uint32_t sbits = mx_scale_bits(m, KIND, rounding);
    const float inv = mx_inv_scale(sbits);
    uint32_t w[BB / 4];
#pragma unroll
    for (int i = 0; i < BB / 4; ++i) w[i] = 0;
    if constexpr (KIND == TK_E2M1) {
      // hardware conversion (round to nearest even, saturating at +-6); NaN is first turned into the infinity of
      // its sign so that it saturates like the reference's bit algorithm (mxfp.py:298-327)
#pragma unroll
      for (int i = 0; i < 32; i += 2) {
        float q0 = elem(i) * inv, q1 = elem(i + 1) * inv;
        q0 = q0 != q0 ? __builtin_copysignf(INFINITY, q0) : q0;
        q1 = q1 != q1 ? __builtin_copysignf(INFINITY, q1) : q1;
        if ((i & 6) == 0) w[i >> 3] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w[i >> 3], q0, q1, 1.0f, 0);
        if ((i & 6) == 2) w[i >> 3] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w[i >> 3], q0, q1, 1.0f, 1);
        if ((i & 6) == 4) w[i >> 3] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w[i >> 3], q0, q1, 1.0f, 2);
        if ((i & 6) == 6) w[i >> 3] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w[i >> 3], q0, q1, 1.0f, 3);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 32; i += 2) w[i >> 2] |= quant_pair<KIND>(elem(i) * inv, elem(i + 1) * inv) << (8 * (i & 2));
    }
#pragma unroll
    for (int i = 0; i < BB / 16; ++i) dst[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    sc_s[(c4 + c) * NB + b] = (uint8_t)(sbits >> 23);
  }
}

// 8 bytes of a stream that is read exactly once: the non-temporal hint (NT) keeps the lines from displacing what the L2
// still has to merge (the output lines at the tiles' seams); measured 0.281 -> 0.264 ms on [32, 2880, 5760] bf16.
// (The same hint on the dequantiser's row stores costs 5 %: 0.275 -> 0.288 ms.)
template <bool NT>
__device__ __forceinline__ uint2 load_once_u2(const uint16_t* p) {
  const u32x2_any_t* a = reinterpret_cast<const u32x2_any_t*>(p);
  const u32x2_any_t t = NT ? __builtin_nontemporal_load(a) : *a;
  return make_uint2(t.x, t.y);
}

// NT: the source is read with the hint; NB: blocks of 32 in a tile (mx_tiles).
template <int SRC, int KIND, bool NT, int NB>
__global__ __launch_bounds__(kThreads) void mx_down_tile(const uint16_t* __restrict__ src, int64_t stride_outer, int64_t stride_axis,
                                                         int64_t L, int64_t inner, int64_t inner_last, int64_t col_tiles,
                                                         int64_t blk_tiles, uint8_t* __restrict__ out_vals,
                                                         uint8_t* __restrict__ out_scales, int rounding) {
  __shared__ __attribute__((aligned(16))) uint8_t vals_s[kTileRows * kTilePitch];
  __shared__ uint8_t sc_s[kTileCols * NB];
  int64_t bid = tile_order(blockIdx.x, gridDim.x);
  const int64_t bt = bid % blk_tiles;
  bid /= blk_tiles;
  const int64_t ct = bid % col_tiles;
  const int64_t o = bid / col_tiles;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: row addresses stay scalar
  const int64_t col0 = tile_col0(ct, inner), blk0 = bt * NB;
  const bool live = col0 + lane * 4 < inner;
  const int c4 = tile_cols_of(lane, col0, inner);  // this lane's four columns inside the tile
  if constexpr (NB / 4 == 2) {
    // e2m1 (two blocks per wave): the rows of BOTH blocks are requested before either is converted.  That takes 171
    // registers, so two workgroups share a CU instead of four, each wave with 32 KB on its way instead of 16: measured
    // 0.314 -> 0.281 ms on [32, 2880, 5760] bf16.  (Fewer resident workgroups help on their own, 0.289 ms with the one-block
    // loop held to two waves per SIMD; one wave per SIMD is too few, 0.317 ms.)
    uint2 raw0[32], raw1[32];
    const bool ok0 = blk0 + wave < L / 32 && live, ok1 = blk0 + wave + 4 < L / 32 && live;
    const int64_t bb0 = ok0 ? blk0 + wave : 0, bb1 = ok1 ? blk0 + wave + 4 : bb0;
    const int64_t cc = live ? col0 + c4 : 0;
    const uint16_t* p0 = src + o * stride_outer + bb0 * 32 * stride_axis + cc;
    const uint16_t* p1 = src + o * stride_outer + bb1 * 32 * stride_axis + cc;
#pragma unroll
    for (int i = 0; i < 32; ++i) raw0[i] = load_once_u2<NT>(p0 + i * stride_axis);
#pragma unroll
    for (int i = 0; i < 32; ++i) raw1[i] = load_once_u2<NT>(p1 + i * stride_axis);
    if (ok0) quantise_block_to_lds<SRC, KIND, NB>(raw0, vals_s, sc_s, c4, wave, rounding);
    if (ok1) quantise_block_to_lds<SRC, KIND, NB>(raw1, vals_s, sc_s, c4, wave + 4, rounding);
  } else
#pragma unroll 1
  for (int pass = 0; pass < NB / 4; ++pass) {
    const int b = wave + 4 * pass;
    if (blk0 + b >= L / 32 || !live) continue;
    const uint16_t* p = src + o * stride_outer + (blk0 + b) * 32 * stride_axis + col0 + c4;
    // the 32 rows stay packed (two 16-bit elements per register) and are widened where they are used: half the
    // registers of an fp32 copy, which is what lets four workgroups share a CU and overlap their load phases
    uint2 raw[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) raw[i] = load_once_u2<NT>(p + i * stride_axis);
    quantise_block_to_lds<SRC, KIND, NB>(raw, vals_s, sc_s, c4, b, rounding);
  }
  __syncthreads();
  tile_store<KIND, NB>(vals_s, sc_s, out_vals, out_scales, o, col0, blk0, L, inner, inner_last);
}

template <int KIND, int DST, int NB, bool TOGETHER>
__global__ __launch_bounds__(kThreads) void mx_up_tile(const uint8_t* __restrict__ vals, const uint8_t* __restrict__ scales, int64_t L,
                                                       int64_t inner, int64_t inner_last, int64_t col_tiles, int64_t blk_tiles,
                                                       uint16_t* __restrict__ out, int64_t ostride_outer, int64_t ostride_axis) {
  constexpr int BB = TileGeom<KIND>::BB;
  __shared__ __attribute__((aligned(16))) uint8_t vals_s[kTileRows * kTilePitch];
  __shared__ uint8_t sc_s[kTileCols * NB];
  int64_t bid = tile_order(blockIdx.x, gridDim.x);
  const int64_t bt = bid % blk_tiles;
  bid /= blk_tiles;
  const int64_t ct = bid % col_tiles;
  const int64_t o = bid / col_tiles;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: row addresses stay scalar
  const int64_t col0 = tile_col0(ct, inner), blk0 = bt * NB;
  const bool live = col0 + lane * 4 < inner;
  const int c4 = tile_cols_of(lane, col0, inner);
  tile_fetch<KIND, NB, TOGETHER>(vals_s, sc_s, vals, scales, o, col0, blk0, L, inner, inner_last);
  __syncthreads();
  const float mf = Elem<DST>::max_finite();
#pragma unroll 1
  for (int pass = 0; pass < NB / 4; ++pass) {
    const int b = wave + 4 * pass;
    if (blk0 + b >= L / 32 || !live) continue;
    uint16_t* q = out + o * ostride_outer + (blk0 + b) * 32 * ostride_axis + col0 + c4;
    // Common case, all four blocks of the lane have a scale for which element * scale is a normal number of the target type whatever the element (fp8:
    // what `up_scale_ok` says, and no NaN or infinity among the codes): the hardware conversion (two codes -> two scaled 16-bit floats, exact, no
    // clamp needed) yields rows (i, i+1) of one column, a byte permute per output dword regroups two columns' results into (column c, column c+1) of one
    // row, and every 8 rows are stored as soon as they are complete.
    uint32_t sb4[4];
    uint4 w4[4][BB / 16];
    bool all_fast = true;
    uint32_t special = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      sb4[c] = sc_s[(c4 + c) * NB + b];
      all_fast = all_fast && up_scale_ok<KIND, DST>(sb4[c]);
      const uint4* srcp = reinterpret_cast<const uint4*>(vals_s + tile_row(c4 + c) * kTilePitch + b * BB);
#pragma unroll
      for (int h = 0; h < BB / 16; ++h) {
        w4[c][h] = srcp[h];
        if constexpr (KIND != TK_E2M1)
          special |= special_codes<KIND>(w4[c][h].x) | special_codes<KIND>(w4[c][h].y) | special_codes<KIND>(w4[c][h].z) | special_codes<KIND>(w4[c][h].w);
      }
    }
    if (all_fast && special == 0) {
      auto word = [](const uint4& v, int k) __attribute__((always_inline)) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; };
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        uint32_t pr[4][4];  // [column][row pair of this group of 8 rows]
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float scale = hd_bits_f32(sb4[c] << 23);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if constexpr (KIND == TK_E2M1)
              pr[c][g] = cvt_pk_from_fp4<DST>(word(w4[c][0], d), scale, g);
            else
              pr[c][g] = cvt_pk_from_8<KIND, DST>(word(w4[c][d >> 1], 2 * (d & 1) + (g >> 1)), scale, g & 1);
          }
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int i = d * 8 + g * 2;
          *reinterpret_cast<u32x2_any_t*>(q + i * ostride_axis) =
              u32x2_any_t{__builtin_amdgcn_perm(pr[1][g], pr[0][g], 0x05040100u), __builtin_amdgcn_perm(pr[3][g], pr[2][g], 0x05040100u)};
          *reinterpret_cast<u32x2_any_t*>(q + (i + 1) * ostride_axis) =
              u32x2_any_t{__builtin_amdgcn_perm(pr[1][g], pr[0][g], 0x07060302u), __builtin_amdgcn_perm(pr[3][g], pr[2][g], 0x07060302u)};
        }
      }
      continue;
    }
    // general path: element by element with the clamp, two rows at a time; a loop, since unrolled over fp8's 128 elements it was most of the time of a
    // small tensor to fetch (2 x 64 x 528 e5m2: 15 to 18 us a launch, 4.5 now; 32 x 2880 x 5760 e4m3 490 us, 345 now, of which the packed conversions are most)
#pragma unroll 1
    for (int i = 0; i < 32; i += 2) {
      uint32_t hp[2][2] = {{0, 0}, {0, 0}};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint8_t* srcp = vals_s + tile_row(c4 + c) * kTilePitch + b * BB;
        const uint32_t sb = sc_s[(c4 + c) * NB + b];
        const uint32_t two = KIND == TK_E2M1 ? srcp[i >> 1] : *reinterpret_cast<const uint16_t*>(srcp + i);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          float f;
          if (KIND == TK_E2M1)
            f = mx_dequant(bf16_bits_to_f32((uint16_t)e2m1_to_bf16_bits((two >> (4 * r)) & 0xFu)), sb, mf, false);
          else
            f = mx_dequant(elem_f32<KIND>((two >> (8 * r)) & 0xFFu), sb, mf, KIND == TK_E5M2);
          uint16_t e;
          Elem<DST>::store(&e, f);
          hp[r][c >> 1] |= (uint32_t)e << (16 * (c & 1));
        }
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) *reinterpret_cast<u32x2_any_t*>(q + (i + r) * ostride_axis) = u32x2_any_t{hp[r][0], hp[r][1]};
    }
  }
}

// ---- dispatch helpers --------------------------------------------------------------------------
template <int SRC, int KIND>
int32_t launch_down(const void* src, int64_t outer, int64_t L, int64_t inner, int64_t inner_last, int64_t so, int64_t sa, int64_t si,
                    void* out_vals, void* out_scales, int rounding, hipStream_t st) {
  typedef typename Elem<SRC>::T T;
  const T* s = static_cast<const T*>(src);
  uint8_t* ov = static_cast<uint8_t*>(out_vals);
  uint8_t* os = static_cast<uint8_t*>(out_scales);
  if (inner == 1 && sa == 1) {
    // rows = outer, row stride = so
    const int64_t total = outer * (L / 8);
    const int64_t grid = cdiv(total, kThreads);
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_downcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_down_rows<SRC, KIND>), dim3((unsigned)grid), dim3(kThreads), 0, st, s, so, outer, L, ov, os,
                       rounding);
    return check_launch("mx_down_rows");
  }
  if (si != 1 && inner != 1) return fail(TK_ERR_UNSUPPORTED, "tk_mx_downcast: inner stride must be 1");
  const int64_t nblk = L / 32;
  const size_t esz = sizeof(T);
  const bool pair_ok = inner % 2 == 0 && sa % 2 == 0 && so % 2 == 0 && (reinterpret_cast<uintptr_t>(src) % (2 * esz)) == 0;
  if constexpr (sizeof(T) == 2) {
    if (inner >= 4 && (reinterpret_cast<uintptr_t>(out_vals) % 16) == 0 && (pair_ok || !mx_by_columns(outer, L, inner))) {
      typedef TileGeom<KIND> G;
      const bool rows8 = inner % 4 == 0 && sa % 4 == 0 && so % 4 == 0 && (reinterpret_cast<uintptr_t>(src) % 8) == 0;
      const MxTiles t = mx_tiles(outer, L, inner, KIND == TK_E2M1, true, rows8);
      if (t.grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_downcast: tensor too large for one launch");
      auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)t.grid), dim3(kThreads), 0, st, reinterpret_cast<const uint16_t*>(s), so, sa, L, inner, inner_last, t.col_tiles, t.blk_tiles, ov, os, rounding);
      };
      if (t.blocks == G::NB)
        launch(t.once ? mx_down_tile<SRC, KIND, true, G::NB> : mx_down_tile<SRC, KIND, false, G::NB>);
      else
        launch(t.once ? mx_down_tile<SRC, KIND, true, G::SMALL> : mx_down_tile<SRC, KIND, false, G::SMALL>);
      return check_launch("mx_down_tile");
    }
  }
  const int64_t blk_tiles = cdiv(nblk, 4);
  if (pair_ok) {
    const int64_t col_tiles = cdiv(inner, 128);
    const int64_t grid = col_tiles * blk_tiles * outer;
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_downcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_down_cols<SRC, KIND, 2>), dim3((unsigned)grid), dim3(kThreads), 0, st, s, so, sa, L, inner,
                       inner_last, col_tiles, blk_tiles, ov, os, rounding);
  } else {
    const int64_t col_tiles = cdiv(inner, 64);
    const int64_t grid = col_tiles * blk_tiles * outer;
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_downcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_down_cols<SRC, KIND, 1>), dim3((unsigned)grid), dim3(kThreads), 0, st, s, so, sa, L, inner,
                       inner_last, col_tiles, blk_tiles, ov, os, rounding);
  }
  return check_launch("mx_down_cols");
}

template <int KIND, int DST>
int32_t launch_up(const void* vals, const void* scales, int64_t outer, int64_t L, int64_t inner, int64_t inner_last, void* out, int64_t oso,
                  int64_t osa, int64_t osi, hipStream_t st) {
  typedef typename Elem<DST>::T T;
  const uint8_t* v = static_cast<const uint8_t*>(vals);
  const uint8_t* s = static_cast<const uint8_t*>(scales);
  T* o = static_cast<T*>(out);
  if (inner == 1 && osa == 1) {
    const int64_t total = outer * (L / 8);
    const int64_t grid = cdiv(total, kThreads);
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_upcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_up_rows<KIND, DST>), dim3((unsigned)grid), dim3(kThreads), 0, st, v, s, outer, L, o, oso);
    return check_launch("mx_up_rows");
  }
  if (osi != 1 && inner != 1) return fail(TK_ERR_UNSUPPORTED, "tk_mx_upcast: output inner stride must be 1");
  const int64_t nblk = L / 32;
  if constexpr (sizeof(T) == 2) {
    if (inner >= 4 && (reinterpret_cast<uintptr_t>(vals) % 16) == 0) {
      typedef TileGeom<KIND> G;
      const MxTiles t = mx_tiles(outer, L, inner, KIND == TK_E2M1, false, false);
      if (t.grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_upcast: tensor too large for one launch");
      auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)t.grid), dim3(kThreads), 0, st, v, s, L, inner, inner_last, t.col_tiles, t.blk_tiles, reinterpret_cast<uint16_t*>(o), oso, osa);
      };
      if (t.blocks == G::SMALL)
        launch(t.together ? mx_up_tile<KIND, DST, G::SMALL, true> : mx_up_tile<KIND, DST, G::SMALL, false>);
      else
        launch(mx_up_tile<KIND, DST, G::NB, false>);
      return check_launch("mx_up_tile");
    }
  }
  const int64_t blk_tiles = cdiv(nblk, 4);
  const size_t esz = sizeof(T);
  const bool pair_ok = inner % 2 == 0 && osa % 2 == 0 && oso % 2 == 0 && (reinterpret_cast<uintptr_t>(out) % (2 * esz)) == 0;
  if (pair_ok) {
    const int64_t col_tiles = cdiv(inner, 128);
    const int64_t grid = col_tiles * blk_tiles * outer;
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_upcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_up_cols<KIND, DST, 2>), dim3((unsigned)grid), dim3(kThreads), 0, st, v, s, L, inner,
                       inner_last, col_tiles, blk_tiles, o, oso, osa);
  } else {
    const int64_t col_tiles = cdiv(inner, 64);
    const int64_t grid = col_tiles * blk_tiles * outer;
    if (grid > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_mx_upcast: tensor too large for one launch");
    hipLaunchKernelGGL((mx_up_cols<KIND, DST, 1>), dim3((unsigned)grid), dim3(kThreads), 0, st, v, s, L, inner,
                       inner_last, col_tiles, blk_tiles, o, oso, osa);
  }
  return check_launch("mx_up_cols");
}

}  // namespace
}  // namespace tk

using namespace tk;

extern "C" int32_t tk_mx_downcast(const void* src, int32_t src_dtype, int64_t outer, int64_t axis_len, int64_t inner,
                                  int64_t inner_last, int64_t stride_outer, int64_t stride_axis, int64_t stride_inner, void* out_vals,
                                  void* out_scales, int32_t out_kind, int32_t rounding, tk_stream_t stream) {
  if (outer < 0 || axis_len < 0 || inner < 0) return fail(TK_ERR_INVALID, "tk_mx_downcast: negative size");
  if (axis_len % 32 != 0) return fail(TK_ERR_INVALID, "tk_mx_downcast: axis length %lld is not a multiple of 32", (long long)axis_len);
  if (rounding != TK_MX_ROUND_UP && rounding != TK_MX_ROUND_DOWN) return fail(TK_ERR_INVALID, "tk_mx_downcast: bad rounding mode %d", rounding);
  if (out_kind != TK_E2M1 && out_kind != TK_E4M3 && out_kind != TK_E5M2) return fail(TK_ERR_INVALID, "tk_mx_downcast: bad output kind %d", out_kind);
  if (outer == 0 || axis_len == 0 || inner == 0) return TK_OK;
  if (inner_last <= 0 || inner % inner_last != 0) return fail(TK_ERR_INVALID, "tk_mx_downcast: inner_last must divide inner");
  if (!src || !out_vals || !out_scales) return fail(TK_ERR_INVALID, "tk_mx_downcast: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define TK_DOWN(S, K) \
  if (src_dtype == S && out_kind == K) return launch_down<S, K>(src, outer, axis_len, inner, inner_last, stride_outer, stride_axis, stride_inner, out_vals, out_scales, rounding, st);
  TK_DOWN(TK_BF16, TK_E2M1)
  TK_DOWN(TK_BF16, TK_E4M3)
  TK_DOWN(TK_BF16, TK_E5M2)
  TK_DOWN(TK_F16, TK_E2M1)
  TK_DOWN(TK_F16, TK_E4M3)
  TK_DOWN(TK_F16, TK_E5M2)
  TK_DOWN(TK_F32, TK_E2M1)
  TK_DOWN(TK_F32, TK_E4M3)
  TK_DOWN(TK_F32, TK_E5M2)
#undef TK_DOWN
  return fail(TK_ERR_INVALID, "tk_mx_downcast: unsupported source dtype %d", src_dtype);
}

extern "C" int32_t tk_mx_upcast(const void* vals, const void* scales, int32_t kind, int64_t outer, int64_t axis_len,
                                int64_t inner, int64_t inner_last, void* out, int32_t out_dtype, int64_t ostride_outer,
                                int64_t ostride_axis, int64_t ostride_inner, tk_stream_t stream) {
  if (outer < 0 || axis_len < 0 || inner < 0) return fail(TK_ERR_INVALID, "tk_mx_upcast: negative size");
  if (axis_len % 32 != 0) return fail(TK_ERR_INVALID, "tk_mx_upcast: axis length %lld is not a multiple of 32", (long long)axis_len);
  if (kind != TK_E2M1 && kind != TK_E4M3 && kind != TK_E5M2) return fail(TK_ERR_INVALID, "tk_mx_upcast: bad element kind %d", kind);
  if (outer == 0 || axis_len == 0 || inner == 0) return TK_OK;
  if (inner_last <= 0 || inner % inner_last != 0) return fail(TK_ERR_INVALID, "tk_mx_upcast: inner_last must divide inner");
  if (!vals || !scales || !out) return fail(TK_ERR_INVALID, "tk_mx_upcast: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
#define TK_UP(K, D) \
  if (kind == K && out_dtype == D) return launch_up<K, D>(vals, scales, outer, axis_len, inner, inner_last, out, ostride_outer, ostride_axis, ostride_inner, st);
  TK_UP(TK_E2M1, TK_BF16)
  TK_UP(TK_E2M1, TK_F16)
  TK_UP(TK_E2M1, TK_F32)
  TK_UP(TK_E4M3, TK_BF16)
  TK_UP(TK_E4M3, TK_F16)
  TK_UP(TK_E4M3, TK_F32)
  TK_UP(TK_E5M2, TK_BF16)
  TK_UP(TK_E5M2, TK_F16)
  TK_UP(TK_E5M2, TK_F32)
#undef TK_UP
  return fail(TK_ERR_INVALID, "tk_mx_upcast: unsupported output dtype %d", out_dtype);
}
