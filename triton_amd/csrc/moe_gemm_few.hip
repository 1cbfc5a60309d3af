// Expert GEMM for few rows per expert with strided, K-contiguous 16-bit weights (bf16 or fp16), fp32 accumulation.
//
//   * A workgroup multiplies up to 64 rows of one slice by 32 or 64 columns.  Its four waves take chunks of 64 k in turn (wave w: chunks w,
//     w + 4, ...) and never wait for one another until their sums meet in LDS: with a tile per workgroup and all of K one after the other
//     (128 x 128 tiles: 16 stages at K 1024, on 32 CUs) the chain was the time.
//   * A chunk comes by `buffer_load ... lds`, eight rows or columns of 128 bytes a transfer, into a ring of the wave's own: three chunks (two
//     with 64 columns) are on their way, 130 to 145 KiB per CU, so a small product is in flight whole.  (Loads in MFMA order straight into
//     registers touch 32 lines for 32 bytes each and took twice the time on the way into the CU.)
//   * Weights are asked for as soon as the slice is known, the gathered rows behind them when their indices have come; rows past the slice,
//     columns past N and k past K are offsets past a resource's end.
//   * Rows are multiplied in fragments of 16 (v_mfma_f32_16x16x32), of which only those with rows are fetched.
//   * A thread sums the waves' parts of four columns of a row, whose bias, gate weight and destination it has loaded before the first chunk.
//
// What bounds it: a chain of latencies (slice sizes, row indices, rows, sums, store), 4.2 us at K 512 with next to nothing to do; its
// instructions come from memory as well, once per launch: with the ring's first turns unrolled and every option of the epilogue in line
// (4900 instructions) the same kernel took 1.2 to 2.3 us longer than now (2300).  Layer of 128 tokens, 8 experts, top 2, d 512,
// d_ff 1024: first GEMM 12.1 -> 9.1 us, second 15.4 -> 7.6 with other weights each call; with the same ones again, as far as they are in the
// caches, 9.4 -> 6.3 and 12.1 -> 5.7.
#include "gemm_common.h"
#include "route_common.h"

namespace tk {
namespace {

template <int BN_>
struct FewCfg {
  static constexpr int BM = 64, BN = BN_, NW = 4;
  static constexpr int WBYTES = BN * 128, XBYTES = BM * 128;  // a chunk of 64 k
  static constexpr int CHUNK = WBYTES + XBYTES;
  static constexpr int BUFS = BN == 32 ? 3 : 2;
  static constexpr int WAVE = BUFS * CHUNK;
  static constexpr int LDS = NW * (WAVE + BM * 4);
  static constexpr int WI = BN / 8;  // transfers of a chunk's weights
  static constexpr int NQ = BM * BN / 4 / (NW * 64);  // results of a thread, four columns each
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// EXTRA: any of the epilogue's options, rows without vector stores, a bias without vector loads.  (The kernel is so short that fetching its
// instructions counts: the common epilogue is compiled by itself.)
template <int BN, bool F16, bool SWIGLU, bool EXTRA>
__global__ __launch_bounds__(256, 1) void moe_gemm_few_kernel(const GemmParams p) {
  typedef FewCfg<BN> C;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, h = lane >> 4;
  const int n0 = blockIdx.y * BN;
  // Row blocks of all slices in order, this workgroup's gridDim.x apart.
  int expert = 0, start_m = 0, eM = p.M, off_m = 0;
  int total = p.slice_sizes ? 0x7FFFFFFF : (p.M + C::BM - 1) / C::BM;  // (with up to 64 slices known from the first search)
  auto locate = [&](int block) __attribute__((always_inline)) -> bool {
    off_m = block * C::BM;
    if (!p.slice_sizes) return true;
#pragma unroll 1
    for (int e0 = 0; e0 < p.n_slices; e0 += 64) {
      int sz = 0, so = 0;
      if (e0 + lane < p.n_slices) {
        sz = p.slice_sizes[e0 + lane];
        so = p.slice_offs[e0 + lane];
      }
      const int cnt = (sz + C::BM - 1) / C::BM, inc = wave_scan_i32(cnt);
      if (p.n_slices <= 64) total = __builtin_amdgcn_readlane(inc, 63);
      const uint64_t over = __builtin_amdgcn_ballot_w64(inc > block);
      if (over) {
        const int l = (int)__builtin_ctzll(over);
        expert = e0 + l;
        eM = __builtin_amdgcn_readlane(sz, l);
        start_m = __builtin_amdgcn_readlane(so, l);
        off_m = (block - (__builtin_amdgcn_readlane(inc, l) - __builtin_amdgcn_readlane(cnt, l))) * C::BM;
        return true;
      }
      block -= __builtin_amdgcn_readlane(inc, 63);
    }
    return false;
  };

  const int N = p.N, KB = p.K * 2;
  const int nch = (p.K + 63) >> 6;
  const int my_chunks = (nch - wave + C::NW - 1) / C::NW;  // chunks wave, wave + 4, ...
  uint8_t* const ring = lds + wave * C::WAVE;
  const uint32_t ring0 = lds_addr(ring), idx0 = lds_addr(lds) + C::NW * C::WAVE + wave * C::BM * 4;
  const buf_desc_t xdesc = make_buf_desc(p.x, p.x_bytes);
  const int cols = N - n0 < BN ? N - n0 : BN;
  const uint32_t x_row = (uint32_t)(p.x_stride_m * 2);
  // transfers: eight rows (columns) of 128 bytes each; lane -> row lane / 8, LDS position lane % 8 holding piece (lane % 8) ^ (row % 8)
  const int t8 = lane >> 3, piece = (lane & 7) ^ t8;
  // (a column past N; with a k past K or without it the sum stays behind every resource here: extents are multiples of 16 below 2 GiB)
  constexpr uint32_t kPastK = 0x7FFFFFF0u;
  uint32_t w_off[C::WI];
#pragma unroll
  for (int q = 0; q < C::WI; ++q) w_off[q] = q * 8 + t8 < cols ? (uint32_t)(q * 8 + t8) * (uint32_t)p.w_stride_n + (uint32_t)piece * 16u : kDroppedStore;
  // fragment reads: row lr, k = t * 32 + h * 8
  uint32_t pos[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) pos[t] = (uint32_t)(lr * 128 + (((t * 4 + h) ^ (lr & 7)) * 16));

  // this thread's results: NQ rows of the same four columns
  constexpr int QW = BN / 4, QR = 256 / QW;
  const int t_cq = tid % QW, t_row = tid / QW, t_n = n0 + t_cq * 4;
  const float nalpha_log2e = -p.alpha * 1.4426950408889634f;
  const float limit = p.has_limit ? p.limit : INFINITY;

  for (int block = blockIdx.x; block < total && locate(block); block += gridDim.x) {
    const int rows = eM - off_m < C::BM ? eM - off_m : C::BM;
    const int first = start_m + off_m;
    const buf_desc_t wdesc = make_buf_desc(p.w + (int64_t)expert * p.w_stride_e + (int64_t)n0 * p.w_stride_n, (uint32_t)(cols - 1) * (uint32_t)p.w_stride_n + (uint32_t)KB);
    // the epilogue's operands, as they lie in memory (a conversion here would wait for them)
    u32x4_t bias_raw = {0, 0, 0, 0};
    if (p.bias && (!EXTRA || p.bias_vec)) {
      const int es = p.bias_is_f32 ? 4 : 2;
      const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(static_cast<const uint8_t*>(p.bias)) + expert * p.bias_stride_e * es, 0, (uint32_t)N * es, 0x00020000);
      if (p.bias_is_f32) {
        bias_raw = __builtin_amdgcn_raw_buffer_load_b128(br, (uint32_t)t_n * 4u, 0, 0);
      } else {
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(br, (uint32_t)t_n * 2u, 0, 0);
        bias_raw[0] = v[0], bias_raw[1] = v[1];
      }
    }
    uint32_t gam_raw[C::NQ];
    int dst_raw[C::NQ];
#pragma unroll
    for (int q = 0; q < C::NQ; ++q) {
      const int r = t_row + q * QR, srow = first + (r < rows ? r : rows - 1);
      gam_raw[q] = 0;
      dst_raw[q] = 0;
      if (p.gammas) gam_raw[q] = p.gammas_is_f32 ? static_cast<const uint32_t*>(p.gammas)[srow] : static_cast<const uint16_t*>(p.gammas)[srow];
      if (p.scatter) dst_raw[q] = p.scatter[srow < p.scatter_len ? srow : p.scatter_len - 1];
    }
    if (p.gather) {
      const buf_desc_t gdesc = make_buf_desc(p.gather + first, (uint32_t)rows * 4u);
      lds_dma4(gdesc, idx0, (uint32_t)lane * 4u);
    }
    // byte offset of k in a row, of this wave's chunk i
    auto k_off = [&](int i) __attribute__((always_inline)) -> uint32_t {
      const uint32_t kb = (uint32_t)(wave + i * C::NW) * 128u;
      return i < my_chunks && (int)kb + piece * 16 < KB ? kb : kPastK;
    };
    auto fetch_w = [&](uint32_t kb, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < C::WI; ++q) lds_dma16(wdesc, to + q * 1024, w_off[q] + kb);
    };
#pragma unroll
    for (int b = 0; b < C::BUFS; ++b) fetch_w(k_off(b), ring0 + b * C::CHUNK);

    auto multiply = [&](auto nj_c) __attribute__((always_inline)) {
      constexpr int NJ = decltype(nj_c)::value;  // row fragments of 16
      constexpr int XI = 2 * NJ, PI = C::WI + XI;
      uint32_t x_off[XI];
      if (p.gather) {
        wait_vm<C::BUFS * C::WI>();
#pragma unroll
        for (int q = 0; q < XI; ++q)
          x_off[q] = *reinterpret_cast<const __attribute__((address_space(3))) uint32_t*>((uintptr_t)(idx0 + (q * 8 + t8) * 4));
      } else {
#pragma unroll
        for (int q = 0; q < XI; ++q) x_off[q] = (uint32_t)(first + q * 8 + t8);
      }
#pragma unroll
      for (int q = 0; q < XI; ++q) x_off[q] = q * 8 + t8 < rows ? x_off[q] * x_row + (uint32_t)piece * 16u : kDroppedStore;
      auto fetch_x = [&](uint32_t kb, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < XI; ++q) lds_dma16(xdesc, to + C::WBYTES + q * 1024, x_off[q] + kb);
      };
#pragma unroll
      for (int b = 0; b < C::BUFS; ++b) fetch_x(k_off(b), ring0 + b * C::CHUNK);
      f32x4_t acc[BN / 16][NJ];
#pragma unroll
      for (int f = 0; f < BN / 16; ++f)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[f][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      uint32_t at = 0;
#pragma unroll 1
      for (int i = 0; i < my_chunks; ++i) {
        // chunk i has landed when only younger transfers are outstanding: of the first chunks all weights came in front of all activations
        static_assert(C::BUFS == 2 || C::BUFS == 3, "the waits below");
        if (i == 0)
          wait_vm<(C::BUFS - 1) * XI>();
        else if (C::BUFS == 3 && i == 1)
          wait_vm<XI + PI>();
        else
          wait_vm<(C::BUFS - 1) * PI>();
        const uint8_t* w = ring + at;
        const uint8_t* x = w + C::WBYTES;
        bf16x8_t wf[BN / 16][2], xf[NJ][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int f = 0; f < BN / 16; ++f) wf[f][t] = *reinterpret_cast<const bf16x8_t*>(w + f * 2048 + pos[t]);
#pragma unroll
          for (int j = 0; j < NJ; ++j) xf[j][t] = *reinterpret_cast<const bf16x8_t*>(x + j * 2048 + pos[t]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint32_t kb = k_off(i + C::BUFS);
        fetch_w(kb, ring0 + at);
        fetch_x(kb, ring0 + at);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int f = 0; f < BN / 16; ++f)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[f][j] = F16 ? Frag<16>::mma_f16(wf[f][t], xf[j][t], acc[f][j]) : Frag<16>::mma(wf[f][t], xf[j][t], acc[f][j]);
        at = at + C::CHUNK == C::BUFS * C::CHUNK ? 0 : at + C::CHUNK;
      }
      wait_vm<0>();  // (what is left are zeros, but into this memory)
#pragma unroll
      for (int f = 0; f < BN / 16; ++f)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int r = j * 16 + lr;
          *reinterpret_cast<f32x4_t*>(ring + (r * QW + ((f * 4 + h) ^ (r & 7))) * 16) = acc[f][j];
        }
    };
    if (rows <= 16)
      multiply(template_int<1>{});
    else if (rows <= 32)
      multiply(template_int<2>{});
    else if (rows <= 48)
      multiply(template_int<3>{});
    else
      multiply(template_int<4>{});
    __syncthreads();
    const int nw = nch < C::NW ? nch : C::NW;
#pragma unroll
    for (int q = 0; q < C::NQ; ++q) {
      const int r = t_row + q * QR;
      if (r >= rows) continue;
      const uint8_t* at = lds + (r * QW + (t_cq ^ (r & 7))) * 16;
      f32x4_t s = *reinterpret_cast<const f32x4_t*>(at);
      for (int w = 1; w < nw; ++w) s += *reinterpret_cast<const f32x4_t*>(at + w * C::WAVE);
      const int srow = first + r;
      const int64_t dst = !p.scatter ? srow : srow < p.scatter_len ? dst_raw[q] : -1;
      if (dst < 0 || t_n >= N) continue;
      const float g = !p.gammas ? 1.f : bits_f32(p.gammas_is_f32 ? gam_raw[q] : gam_raw[q] << 16);
      const float beta = EXTRA && p.betas ? load_scalar(p.betas, srow, p.betas_is_f32) : 1.f;
      const float rsc = EXTRA && p.x_row_scale ? p.x_row_scale[p.gather ? p.gather[srow] : srow] : 1.f;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = t_n + i < N ? t_n + i : N - 1;
        v[i] = s[i];
        if (EXTRA && (p.x_row_scale || p.w_col_scale)) v[i] *= rsc * (p.w_col_scale ? p.w_col_scale[expert * p.wcs_stride_e + n] : 1.f);
        if (p.bias) {
          const float b = EXTRA && !p.bias_vec ? load_scalar(p.bias, expert * p.bias_stride_e + n, p.bias_is_f32)
                          : p.bias_is_f32 ? bits_f32(bias_raw[i]) : bits_f32(i & 1 ? bias_raw[i >> 1] & 0xFFFF0000u : bias_raw[i >> 1] << 16);
          v[i] = EXTRA && p.betas ? fmaf(b, beta, v[i]) : v[i] + b;
        }
        if (EXTRA && p.has_out_alpha) v[i] *= p.out_alpha;
      }
      constexpr int NV = SWIGLU ? 2 : 4;
      const int o0 = SWIGLU ? t_n / 2 : t_n, n_out = SWIGLU ? N / 2 : N;
      float o[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) o[i] = (SWIGLU ? swiglu_f(v[2 * i & 3], v[(2 * i + 1) & 3], nalpha_log2e, limit) : v[i]) * g;
      uint16_t* y = p.y + dst * p.y_stride_m + o0;
      if (EXTRA && p.acc_in) {
        const uint16_t* a = p.acc_in + dst * p.acc_in_stride_m + o0;
#pragma unroll
        for (int i = 0; i < NV; ++i)
          if (o0 + i < n_out) o[i] += F16 ? f16_bits_to_f32(a[i]) : bf16_bits_to_f32(a[i]);
      }
      if (!EXTRA || (p.y_vec && o0 + NV <= n_out)) {
        uint32_t u[NV / 2];
#pragma unroll
        for (int i = 0; i < NV / 2; ++i) u[i] = pack_out2<F16>(o[2 * i], o[2 * i + 1]);
        if constexpr (SWIGLU)
          *reinterpret_cast<uint32_t*>(y) = u[0];
        else
          *reinterpret_cast<uint2*>(y) = make_uint2(u[0], u[NV / 2 - 1]);
      } else {
#pragma unroll
        for (int i = 0; i < NV; ++i)
          if (o0 + i < n_out) y[i] = cvt_out<F16>(o[i]);
      }
    }
    __syncthreads();
  }
}

template <int BN>
int32_t launch_few(const GemmParams& p, int wk, bool swiglu, hipStream_t st) {
  typedef FewCfg<BN> C;
  const int64_t tiles_n = cdiv(p.N, BN);
  const int64_t n = p.slice_sizes ? p.n_slices : 1, blocks = p.slice_sizes ? few_row_blocks(p.M, n) : cdiv(p.M, C::BM);
  if (n == 0) return TK_OK;
  if (tiles_n > 65535) return fail(TK_ERR_UNSUPPORTED, "tk_moe_gemm: grid too large");
  auto launch = [&](auto kern) -> int32_t {
    if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), C::LDS)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, (unsigned)tiles_n), dim3(C::NW * 64), C::LDS, st, p);
    return check_launch("moe_gemm_few_kernel");
  };
  const bool extra = p.x_row_scale || p.w_col_scale || p.betas || p.has_out_alpha || p.acc_in || !p.y_vec || p.N % 4 || (p.bias && !p.bias_vec);
  auto with = [&](auto f16, auto act) -> int32_t {
    constexpr bool F16 = decltype(f16)::value, SWIGLU = decltype(act)::value;
    return extra ? launch(moe_gemm_few_kernel<BN, F16, SWIGLU, true>) : launch(moe_gemm_few_kernel<BN, F16, SWIGLU, false>);
  };
  const std::true_type yes;
  const std::false_type no;
  if (wk == WK_F16) return swiglu ? with(yes, yes) : with(yes, no);
  return swiglu ? with(no, yes) : with(no, no);
}

}  // namespace

int32_t gemm_launch_few(const GemmParams& p, int wk, int block_n, bool swiglu, hipStream_t st) {
  return block_n == 64 ? launch_few<64>(p, wk, swiglu, st) : launch_few<32>(p, wk, swiglu, st);
}

}  // namespace tk
