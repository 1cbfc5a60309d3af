// The decode layer (moe_decode_layer.hip) row by row, in two launches, for small streams of weights (the entry point says which).
//
//   * Launch 1: a workgroup of eight waves = one routed row x 32 columns of W1.  It selects its own token's experts (every wave for itself, a
//     row of logits), so no launch and no table stands in front of the weights; its waves take the K-stages in turn, each with all of its
//     weights requested at once (at K 2880 6 KiB), and meet in LDS once.  Up to four workgroups share a CU: 200 KiB of weights on their way.
//   * Launch 2: a workgroup of sixteen waves = one token x 16 columns of W2 for ALL of the token's experts, so that the sum over the experts
//     needs neither counters nor another launch.
//   * The row lies in LDS, from where every lane of a k-group reads the same bytes: the MFMA's sixteen rows are one row sixteen times, which
//     costs nothing beside the stream.
//
// What bounds it: launch 1 two dependent trips to memory (logits, weights) and launch 2 two (table, weights) around the streams of 35 and
// 18 MB.  One token, 4 of 128 experts, K 2880, N 5760 and 2880: 17.9 us (ten such layers in a graph, one after the
// other); with routing, a GEMM, and a GEMM that counts its rows for the sum as launches of their own 28.4 us.
#include "decode_params.h"
#include "gemm_common.h"
#include "route_common.h"

namespace tk {
namespace {

constexpr int kMaxStages = 24;  // K <= 3072
constexpr int kMaxK = kDecRowsMaxK;
struct RowEntry {
  int32_t expert;
  float gate;
};

// This lane's 16 bytes of columns g * 16 + lr (of a fragment of 32) and k-block kg of a stage, and the columns' scales.
template <bool ONCE>
struct Piece {
  u32x4_t w;
  uint32_t s;
  __device__ __forceinline__ void load(const uint8_t* w_at, const uint8_t* s_at) {
    if constexpr (ONCE) {
      w = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(w_at));
      s = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(s_at));
    } else {
      w = *reinterpret_cast<const u32x4_t*>(w_at);
      s = *reinterpret_cast<const uint32_t*>(s_at);
    }
  }
  // row: the stage's 128 k of the row in LDS (every lane of a k-group reads the same bytes)
  __device__ __forceinline__ f32x4_t times(const uint8_t* row, int kg, f32x4_t acc) const {
    const float scale = bits_f32(((s >> (8 * kg)) & 0xFFu) << 23);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      acc = Frag<16>::mma(dequant8(w[t], scale), *reinterpret_cast<const bf16x8_t*>(row + kg * 64 + t * 16), acc);
    return acc;
  }
};

// Rows of K bf16 values, `stride` elements apart, into LDS, each padded with zeros to nst stages.
__device__ __forceinline__ void stage_rows(uint8_t* dst, const uint16_t* src, int64_t stride, int rows, int K, int nst, int threads) {
  const int per = nst * 16;
  for (int i = threadIdx.x; i < rows * per; i += threads) {
    const int r = i / per, c = (i - r * per) * 8;
    u32x4_t v = {0, 0, 0, 0};
    if (c < K) v = *reinterpret_cast<const u32x4_t*>(src + r * stride + c);
    *reinterpret_cast<u32x4_t*>(dst + (size_t)i * 16) = v;
  }
}

// Launch 1: blockIdx.y = routed row t * k + j, blockIdx.x = 32 columns of W1.  Every workgroup selects its token's experts itself.
constexpr int kUpWaves = 8, kUpStages = kMaxStages / kUpWaves;
template <int EPL, bool ONCE>
__global__ __launch_bounds__(kUpWaves * 64) void decode_rows_up_kernel(const DecodeParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t x_s[kMaxStages * 256];
  __shared__ __attribute__((aligned(16))) float part_s[kUpWaves][32];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, kg = lane >> 4;
  const int row = blockIdx.y, t = row / p.k, j = row - t * p.k, F = blockIdx.x;
  float v[EPL];
  {
    const int64_t at = (int64_t)t * p.logits_stride;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int e = lane + 64 * i < p.E ? lane + 64 * i : p.E - 1;
      v[i] = p.logits_is_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(p.logits)[at + e]) : static_cast<const float*>(p.logits)[at + e];
    }
  }
  stage_rows(x_s, reinterpret_cast<const uint16_t*>(p.x) + t * p.x_stride, 0, 1, p.K1, p.nst1, kUpWaves * 64);
  uint32_t key[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) key[i] = lane + 64 * i < p.E ? ordered_key(v[i]) : 0u;
  float top_v = 0.f;
  int top_e = -1;
  wave_topk<EPL>(key, p.k, p.E, lane, top_v, top_e);
  const int expert = __builtin_amdgcn_readlane(top_e, j);

  // this wave's stages: wave, wave + 8, ...
  Piece<ONCE> piece[kUpStages][2];
  {
    const uint8_t* w = p.w1 + (int64_t)expert * p.w1_stride_e + (int64_t)F * p.nst1 * 2048 + (kg & 1) * 1024 + ((kg >> 1) * 32 + lr) * 16;
    const uint8_t* s = p.w1s + (int64_t)expert * p.w1s_stride_e + (int64_t)F * p.nst1 * 128 + lr * 4;
#pragma unroll
    for (int i = 0; i < kUpStages; ++i) {
      const int st = wave + i * kUpWaves < p.nst1 ? wave + i * kUpWaves : p.nst1 - 1;
#pragma unroll
      for (int g = 0; g < 2; ++g) piece[i][g].load(w + (int64_t)st * 2048 + g * 256, s + (int64_t)st * 128 + g * 64);
    }
  }
  const int n = F * 32 + threadIdx.x;  // (threads 0 to 31: the column that they finish)
  float bias = 0.f;
  if (threadIdx.x < 32 && p.b1 && n < p.N1) bias = load_scalar(p.b1, expert * p.b1_stride_e + n, p.b1_is_f32);
  if (F == 0 && wave == 0 && j == 0) {
    // the token's gate values, for the second launch and for whoever asks for them
    float gate = top_v;
    if (p.apply_softmax) {
      const float vmax = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, top_v), 0));
      const float z = lane < p.k ? expf(top_v - vmax) : 0.f;
      gate = z / wave_sum_f32(z);
    }
    if (lane < p.k) {
      if (p.indx_out) p.indx_out[(int64_t)t * p.k + lane] = (int16_t)top_e;
      if (p.vals_out) p.vals_out[(int64_t)t * p.k + lane] = gate;
      reinterpret_cast<RowEntry*>(p.y)[t * p.k + lane] = RowEntry{top_e, gate};
    }
  }
  __syncthreads();
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < kUpStages; ++i) {
    const int st = wave + i * kUpWaves;
    if (st < p.nst1) {
#pragma unroll
      for (int g = 0; g < 2; ++g) acc[g] = piece[i][g].times(x_s + st * 256, kg, acc[g]);
    }
  }
  // (all sixteen rows of the fragment are the same row: lane lr 0 of every k-group holds four columns' sums)
  if (lr == 0) {
#pragma unroll
    for (int g = 0; g < 2; ++g) *reinterpret_cast<f32x4_t*>(&part_s[wave][g * 16 + kg * 4]) = acc[g];
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kUpWaves; ++w) sum += part_s[w][threadIdx.x];
    sum += bias;
    const float lin = __shfl_xor(sum, 1);
    const float o = swiglu_f(sum, lin, -p.alpha * 1.4426950408889634f, p.has_limit ? p.limit : INFINITY);
    if (!(threadIdx.x & 1) && n < p.N1) p.h[(int64_t)row * p.K2 + n / 2] = f32_to_bf16_bits(o);
  }
}

// Launch 2: blockIdx.y = token, blockIdx.x = 16 columns of W2 for all of the token's experts, so that the workgroup sums them.
constexpr int kDownWaves = 16, kDownStages = 6;
template <bool ONCE>
__global__ __launch_bounds__(kDownWaves * 64) void decode_rows_down_kernel(const DecodeParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t h_s[kMaxK * kMaxStages * 256];
  __shared__ __attribute__((aligned(16))) float part_s[kDownWaves][16];
  __shared__ float y_s[kMaxK][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, kg = lane >> 4;
  const int t = blockIdx.y, n0 = blockIdx.x * 16, F = blockIdx.x >> 1, g = blockIdx.x & 1, k = p.k;
  // the waves share the token's experts evenly, an expert's waves take its stages in turn
  const int per = kDownWaves / k, j = wave / per, part = wave - j * per;
  const RowEntry* table = reinterpret_cast<const RowEntry*>(p.y) + t * k;
  const int expert = __builtin_amdgcn_readfirstlane(j < k ? table[j].expert : 0);
  // this thread's result: column c of expert tj
  const int tj = threadIdx.x >> 4, c = threadIdx.x & 15;
  RowEntry mine = {0, 0.f};
  float bias = 0.f;
  if (tj < k) mine = table[tj];
  const int nst = p.nst2;
  const uint8_t* w = p.w2 + (int64_t)expert * p.w2_stride_e + (int64_t)F * nst * 2048 + g * 256 + (kg & 1) * 1024 + ((kg >> 1) * 32 + lr) * 16;
  const uint8_t* s = p.w2s + (int64_t)expert * p.w2s_stride_e + (int64_t)F * nst * 128 + g * 64 + lr * 4;
  Piece<ONCE> piece[kDownStages];
  auto load = [&](int first) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kDownStages; ++i) {
      int st = part + (first + i) * per;
      st = st < nst ? st : nst - 1;
      piece[i].load(w + (int64_t)st * 2048, s + (int64_t)st * 128);
    }
  };
  if (j < k) load(0);
  stage_rows(h_s, p.h + (int64_t)t * k * p.K2, p.K2, k, p.K2, nst, kDownWaves * 64);
  if (tj < k && p.b2 && n0 + c < p.N2) bias = load_scalar(p.b2, mine.expert * p.b2_stride_e + n0 + c, p.b2_is_f32);
  __syncthreads();
  if (j < k) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int first = 0;;) {
#pragma unroll
      for (int i = 0; i < kDownStages; ++i) {
        const int st = part + (first + i) * per;
        if (st < nst) acc = piece[i].times(h_s + (size_t)(j * nst + st) * 256, kg, acc);
      }
      first += kDownStages;
      if (part + first * per >= nst) break;
      load(first);
    }
    if (lr == 0) *reinterpret_cast<f32x4_t*>(&part_s[wave][kg * 4]) = acc;
  }
  __syncthreads();
  if (tj < k) {
    float sum = 0.f;
    for (int w2 = 0; w2 < per; ++w2) sum += part_s[tj * per + w2][c];
    // (rounded as the row of a GEMM's result is before the sum over the experts)
    y_s[tj][c] = bf16_bits_to_f32(f32_to_bf16_bits((sum + bias) * mine.gate));
  }
  __syncthreads();
  if (threadIdx.x < 16 && n0 + threadIdx.x < p.N2) {
    float sum = 0.f;
    for (int i = 0; i < k; ++i) sum += y_s[i][threadIdx.x];
    p.out[(int64_t)t * p.out_stride + n0 + threadIdx.x] = f32_to_bf16_bits(sum);
  }
}

}  // namespace

int32_t decode_launch_rows(const DecodeParams& p, hipStream_t st) {
  const dim3 up((unsigned)p.nfr1, (unsigned)(p.T * p.k)), down((unsigned)cdiv(p.N2, 16), (unsigned)p.T);
  auto launch = [&](auto up_kern, auto down_kern) -> int32_t {
    // the two launches of a call stay together: another thread's on the same stream may have the same workspace
    static std::mutex together;
    std::lock_guard<std::mutex> lock(together);
    hipLaunchKernelGGL(up_kern, up, dim3(kUpWaves * 64), 0, st, p);
    if (const int32_t rc = check_launch("decode_rows_up_kernel")) return rc;
    hipLaunchKernelGGL(down_kern, down, dim3(kDownWaves * 64), 0, st, p);
    return check_launch("decode_rows_down_kernel");
  };
  // (one token: its experts differ, every weight byte is read once)
  const bool once = p.T == 1;
  if (p.E <= 128) return once ? launch(decode_rows_up_kernel<2, true>, decode_rows_down_kernel<true>) : launch(decode_rows_up_kernel<2, false>, decode_rows_down_kernel<false>);
  return once ? launch(decode_rows_up_kernel<8, true>, decode_rows_down_kernel<true>) : launch(decode_rows_up_kernel<8, false>, decode_rows_down_kernel<false>);
}

}  // namespace tk
