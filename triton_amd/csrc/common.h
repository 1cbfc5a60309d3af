// Shared declarations for the gfx950 kernels behind the C ABI of include/triton_amd.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/triton_amd.h"

namespace tk {

// Records a message for tk_last_error() and returns `code`.
int32_t fail(int32_t code, const char* fmt, ...);

inline int32_t check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TK_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
  return TK_OK;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;

// ---- scalar conversions usable on host and device --------------------------------------------
__host__ __device__ inline float bf16_bits_to_f32(uint16_t b) {
  uint32_t u = (uint32_t)b << 16;
  float f;
  __builtin_memcpy(&f, &u, 4);
  return f;
}

// fp32 -> bf16 bits, round to nearest even, NaN kept quiet (same as torch's cast).
__host__ __device__ inline uint16_t f32_to_bf16_bits(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x0040u);
  uint32_t r = 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)((u + r) >> 16);
}

__device__ inline float f16_bits_to_f32(uint16_t b) {
  _Float16 h;
  __builtin_memcpy(&h, &b, 2);
  return (float)h;
}

__device__ inline uint16_t f32_to_f16_bits(float f) {
  _Float16 h = (_Float16)f;
  uint16_t b;
  __builtin_memcpy(&b, &h, 2);
  return b;
}

// ---- memory straight into LDS ------------------------------------------------------------------
// `u32x4` buffer resource over [base, base + bytes): loads past the range read zero.
typedef uint32_t buf_desc_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ buf_desc_t make_buf_desc(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return buf_desc_t{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
// 16 bytes per lane from `desc` at byte offset `off` into LDS at `dst` (wave-uniform byte address) + 16 * lane.  Written
// as assembly because the compiler puts a wait for ALL outstanding memory operations in front of every LDS read that
// follows the builtin form; here the kernel places its own vmcnt waits (the instruction counts as one).  m0, from which the transfer takes
// its LDS address, is an operand, so that the compiler knows of it and computes the address straight into it.
// Wait states: a vector memory instruction may read a scalar register no sooner than five wait states after a vector instruction wrote it, and the
// compiler, which keeps that distance for its own instructions, does not look into assembly.  A descriptor's words come from v_readfirstlane, or
// back from a spill by v_readlane, at whatever distance the scheduler likes (two in one kernel: its first transfers now and then went by the
// register's old contents, and read zeros or past the operand).  So a transfer reads copies that scalar moves of its own have made, which wait for such a
// write by themselves.  The two moves are also the wait state that a write of m0 needs.  (Five idle states in front of each transfer instead: 300
// tokens of 128 MXFP4 experts, K 2880, layer 319 us against 316; 8192 of 8 in e4m3, K 4096 and 14336, 2611 against 2569.)
// NT = with the non-temporal hint (streams that are read once).
#define TK_DMA_DESC "s_mov_b64 s[92:93], %[lo]\n\ts_mov_b64 s[94:95], %[hi]\n\t"
#define TK_DMA_ARGS(desc) [lo] "s"(desc_half(desc, 0)), [hi] "s"(desc_half(desc, 1))
#define TK_DMA_USED "memory", "s92", "s93", "s94", "s95"
__device__ __forceinline__ uint64_t desc_half(buf_desc_t d, int i) { return (uint64_t)d[2 * i + 1] << 32 | d[2 * i]; }
template <bool NT = false>
__device__ __forceinline__ void lds_dma16(buf_desc_t desc, uint32_t dst, uint32_t off) {
  if constexpr (NT)
    asm volatile(TK_DMA_DESC "buffer_load_dwordx4 %[o], s[92:95], 0 offen nt lds" ::"{m0}"(dst), [o] "v"(off), TK_DMA_ARGS(desc) : TK_DMA_USED);
  else
    asm volatile(TK_DMA_DESC "buffer_load_dwordx4 %[o], s[92:95], 0 offen lds" ::"{m0}"(dst), [o] "v"(off), TK_DMA_ARGS(desc) : TK_DMA_USED);
}
// the same by the lower 32 lanes only (512 bytes; every lane is active when it is called)
__device__ __forceinline__ void lds_dma16_lower(buf_desc_t desc, uint32_t dst, uint32_t off) {
  asm volatile(TK_DMA_DESC "s_mov_b32 exec_hi, 0\n\tbuffer_load_dwordx4 %[o], s[92:95], 0 offen lds\n\ts_mov_b32 exec_hi, -1" ::"{m0}"(dst), [o] "v"(off),
               TK_DMA_ARGS(desc) : TK_DMA_USED);
}
// the same with 4 bytes per lane
template <bool NT = false>
__device__ __forceinline__ void lds_dma4(buf_desc_t desc, uint32_t dst, uint32_t off) {
  if constexpr (NT)
    asm volatile(TK_DMA_DESC "buffer_load_dword %[o], s[92:95], 0 offen nt lds" ::"{m0}"(dst), [o] "v"(off), TK_DMA_ARGS(desc) : TK_DMA_USED);
  else
    asm volatile(TK_DMA_DESC "buffer_load_dword %[o], s[92:95], 0 offen lds" ::"{m0}"(dst), [o] "v"(off), TK_DMA_ARGS(desc) : TK_DMA_USED);
}
// A stage of two MXFP4 fragments: 4 KiB of values (the first fragment's two KiB at `off`, the second's at `off1`, less the 2 KiB that they lie
// behind in LDS: an instruction's offset counts on both sides), then their scales, 4 bytes per lane.  One copy of each descriptor and two writes of m0
// for five transfers.
#define TK_DMA_MXFP4(nt)                                                                                                                     \
  "buffer_load_dwordx4 %[o], s[92:95], 0 offen" nt " lds\n\tbuffer_load_dwordx4 %[o], s[92:95], 0 offen offset:1024" nt                         \
  " lds\n\tbuffer_load_dwordx4 %[p], s[92:95], 0 offen offset:2048" nt " lds\n\tbuffer_load_dwordx4 %[p], s[92:95], 0 offen offset:3072" nt        \
  " lds\n\ts_add_u32 m0, m0, 0x1000\n\ts_mov_b64 s[92:93], %[slo]\n\ts_mov_b64 s[94:95], %[shi]\n\tbuffer_load_dword %[q], s[92:95], 0 offen" nt " lds"
template <bool NT>
__device__ __forceinline__ void lds_dma_mxfp4(buf_desc_t wdesc, buf_desc_t sdesc, uint32_t dst, uint32_t off, uint32_t off1, uint32_t s_off) {
  if constexpr (NT)
    asm volatile(TK_DMA_DESC TK_DMA_MXFP4(" nt") : "+{m0}"(dst) : [o] "v"(off), [p] "v"(off1), [q] "v"(s_off), TK_DMA_ARGS(wdesc),
                 [slo] "s"(desc_half(sdesc, 0)), [shi] "s"(desc_half(sdesc, 1)) : TK_DMA_USED, "scc");
  else
    asm volatile(TK_DMA_DESC TK_DMA_MXFP4("") : "+{m0}"(dst) : [o] "v"(off), [p] "v"(off1), [q] "v"(s_off), TK_DMA_ARGS(wdesc),
                 [slo] "s"(desc_half(sdesc, 0)), [shi] "s"(desc_half(sdesc, 1)) : TK_DMA_USED, "scc");
}
#undef TK_DMA_MXFP4
#undef TK_DMA_DESC
#undef TK_DMA_ARGS
#undef TK_DMA_USED
// LDS byte address of a __shared__ object
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p);
}
// four consecutive k of this lane's row, transposed by the LDS read: sixteen lanes read four rows (lane >> 2 of the group) of
// sixteen 16-bit columns (four per lane) and lane i receives column i of the four rows
__device__ __forceinline__ uint64_t lds_read_tr16(uint32_t at) {
  typedef __attribute__((ext_vector_type(4))) short s16x4_t;
  return __builtin_bit_cast(uint64_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<__attribute__((address_space(3))) s16x4_t*>((uintptr_t)at)));
}

__device__ inline uint32_t f32_bits(float f) { return __builtin_bit_cast(uint32_t, f); }
__device__ inline float bits_f32(uint32_t u) { return __builtin_bit_cast(float, u); }

}  // namespace tk
