// Expert GEMM, bf16 x tiled MXFP4, for row blocks of up to 32 rows: a stream of the active experts' weights, each byte read once.  It serves what the wide
// kernel (moe_gemm_mxw_kernel.h), 1 to 10 % faster at these sizes, does not take: fewer than four stages of K, output rows of no multiple of eight columns.
//
//   * A workgroup multiplies the (up to) 32 rows of one row block by 256 columns: each of its four waves owns two 32-column weight fragments
//     and all rows.  The rows' activations are fetched once per workgroup and stage and shared through LDS (in a kernel in which every wave
//     fetches its own rows they are as many bytes as the weights of two fragments, on the same path into the CU).
//   * A stage is 128 k: 4 KiB + 256 bytes of weights and scales per wave, 256 bytes per row.  All of it comes by `buffer_load ... lds` into a ring
//     of three stages: no registers wait for memory, 100 KiB per CU are on their way at any time, and rows past the slice, columns past N and k
//     past K are a matter of the lanes' offsets (past the resource's range the hardware writes zeros).
//   * e2m1 -> bf16 in registers (v_cvt_scalef32_pk_bf16_fp4) in front of v_mfma_f32_32x32x16_bf16, transposed like the other kernels.
//   * Persistent workgroups, two per CU; the ring runs on across tiles.
//
// What bounds it: reading the weights, 5.1 to 5.4 TB/s at 300 tokens with the matrix pipe 35 % busy.  128 experts, K = 2880, 8 routed rows per expert and more (300 tokens, top-4): N 5760 232 ->
// 210 us, N 2880 149 -> 115 us against the decode kernel; 18 rows: 340 -> 245 and 211 -> 128 us.  More rows multiply more than they stream: at
// 31 rows the prefill kernel's 64-row blocks win (290 against 331 us).  Measured and left out: 64-row blocks (slower than both from 8 to 31
// rows), two or four stages in the ring (no difference).
#include "gemm_tiles.h"

namespace tk {
namespace {

struct MxsCfg {
  static constexpr int MFW = 1, NW = 4;     // row fragments, waves
  static constexpr int BM = MFW * 32, BN = NW * 64;
  static constexpr int ABYTES = BM * 256;
  static constexpr int WBYTES = 4096 + 256;  // a wave's two fragments: values, scales
  static constexpr int STAGE = ABYTES + NW * WBYTES;
  static constexpr int BUFS = 3;
  static constexpr int LDS = BUFS * STAGE;
  static constexpr int AI = BM / 4 / NW;     // activation transfers (four rows each) of a wave and stage
  static constexpr int PI = AI + 5;
};

// ONCE: few slices have several row blocks, so the weights are read about once: fetched with the non-temporal hint
template <bool SWIGLU, bool ONCE>
__global__ __launch_bounds__(MxsCfg::NW * 64, 2) void moe_gemm_mxs_kernel(const GemmParams p) {
  typedef MxsCfg C;
  constexpr int MFW = C::MFW;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;
  const int nst = p.w_nst;
  const uint32_t lds0 = lds_addr(lds);

  TileList<C::BM, C::BN> tiles;
  int tile = tiles.init(p, lane, p.grid_n);
  const int t_step = tiles.t_step, t_end = tiles.t_end;
  if (tile >= t_end) return;

  // ---- transfer side ------------------------------------------------------------------------------------------------------------------------------
  // activations: transfer i = rows (wave * AI + i) * 4 .. + 3, lane -> row lane / 16, LDS position lane % 16 holding piece (lane % 16) ^ (row % 16)
  const buf_desc_t xdesc = make_buf_desc(p.x, p.x_bytes);
  buf_desc_t wdesc, sdesc;
  uint32_t a_off[C::AI];
  int a_k[C::AI];  // first k of the lane's piece
#pragma unroll
  for (int i = 0; i < C::AI; ++i) a_k[i] = ((lane & 15) ^ ((((wave * C::AI + i) & 3) << 2) | (lane >> 4))) * 8;
  const uint32_t x_row = (uint32_t)(p.x_stride_m * 2);
  const int nfr = (p.N + 31) >> 5;
  const uint32_t f_val = (uint32_t)nst * 2048u, f_scale = (uint32_t)nst * 128u;  // bytes of a fragment
  const uint32_t w_off = (uint32_t)lane * 16u, s_off = (uint32_t)(lane >> 5) * f_scale + (uint32_t)lr * 4u;
  auto aim = [&](const Tile& c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::AI; ++i) {
      const int row = c.off_m + (wave * C::AI + i) * 4 + (lane >> 4);
      const int sr = c.start_m + (row < c.eM ? row : c.eM - 1);
      const uint32_t src = p.gather ? (uint32_t)p.gather[sr] : (uint32_t)sr;
      a_off[i] = row < c.eM ? src * x_row + (uint32_t)a_k[i] * 2u : kOutOfRange;
    }
    // this wave's two fragments; past the last one nothing is in range (zeros: the columns are not stored)
    const int f0 = (c.n_tile >> 5) + wave * 2;
    const int nf = nfr - f0 < 0 ? 0 : nfr - f0 < 2 ? nfr - f0 : 2;
    wdesc = make_buf_desc(p.w + (int64_t)c.expert * p.w_stride_e + (int64_t)f0 * f_val, (uint32_t)nf * f_val);
    sdesc = make_buf_desc(p.w_scale + (int64_t)c.expert * p.ws_stride_e + (int64_t)f0 * f_scale, (uint32_t)nf * f_scale);
  };
  auto fetch = [&](int s, uint32_t buf, bool more) __attribute__((always_inline)) {
    const uint32_t wdst = lds0 + buf + C::ABYTES + wave * C::WBYTES;
    const uint32_t at = w_off + (uint32_t)s * 2048u;
    lds_dma_mxfp4<ONCE>(wdesc, sdesc, wdst, more ? at : kOutOfRange, more ? at + (f_val - 2048u) : kOutOfRange, more ? s_off + (uint32_t)s * 128u : kOutOfRange);
#pragma unroll
    for (int i = 0; i < C::AI; ++i)
      lds_dma16(xdesc, lds0 + buf + (wave * C::AI + i) * 1024, more && s * 128 + a_k[i] < p.K ? a_off[i] + (uint32_t)s * 256u : kOutOfRange);
  };

  // ---- the ring: one cursor, two stages ahead of the multiplication -----------------------------------------------------------------------------
  constexpr uint32_t kEnd = C::BUFS * C::STAGE;
  Tile cur = tiles.locate(tile);
  aim(cur);
  uint32_t wb = 0, rb = 0;  // buffers the next transfers fill / the next stage is read from
  int fs = 0, f_tile = tile;
  bool more = true;
  auto advance = [&]() __attribute__((always_inline)) {
    wb = wb + C::STAGE == kEnd ? 0 : wb + C::STAGE;
    if (++fs == nst) {
      fs = 0;
      f_tile += t_step;
      more = more && f_tile < t_end;
      if (more) aim(tiles.locate(f_tile));
    }
  };
  fetch(fs, wb, more);
  advance();
  fetch(fs, wb, more);
  advance();

  f32x16_t acc[2][MFW];
  while (true) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int j = 0; j < MFW; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[f][j][i] = 0.f;
    for (int s = 0; s < nst; ++s) {
      // stage s has landed (this wave's part) when only the transfers of stage s + 1 are outstanding; the buffer of stage s - 1 has been read
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(C::PI) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      fetch(fs, wb, more);
      const uint8_t* a = lds + rb + lr * 256;
      const uint8_t* w = lds + rb + C::ABYTES + wave * C::WBYTES;
      u32x4_t raw[2][2];
      uint32_t sc[2];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        sc[f] = *reinterpret_cast<const uint32_t*>(w + 4096 + f * 128 + lr * 4);
#pragma unroll
        for (int q = 0; q < 2; ++q) raw[f][q] = *reinterpret_cast<const u32x4_t*>(w + f * 2048 + q * 1024 + lane * 16);
      }
      // step t: lane half h supplies k = h * 64 + t * 8 .. + 7, which lie in MX block 2h + t / 4 of the stage
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        bf16x8_t xf[MFW];
#pragma unroll
        for (int j = 0; j < MFW; ++j) xf[j] = *reinterpret_cast<const bf16x8_t*>(a + j * 8192 + (((h * 8 + t) ^ (lr & 15)) * 16));
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          const bf16x8_t wf = dequant8(raw[f][t >> 2][t & 3], bits_f32(((sc[f] >> (16 * h + 8 * (t >> 2))) & 0xFFu) << 23));
#pragma unroll
          for (int j = 0; j < MFW; ++j) acc[f][j] = Frag<32>::mma(wf, xf[j], acc[f][j]);
        }
      }
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int j = 0; j < MFW; ++j) asm volatile("" : "+v"(acc[f][j]));
      rb = rb + C::STAGE == kEnd ? 0 : rb + C::STAGE;
      advance();
    }
    gemm_epilogue<32, 1, MFW, 2, SWIGLU>(p, acc, cur.expert, cur.off_m, cur.start_m, cur.eM, cur.n_tile + wave * 64, cur.n_tile + C::BN <= p.N, 0, lr, h);
    tile += t_step;
    if (tile >= t_end) break;
    cur = tiles.locate(tile);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into this workgroup's LDS is left behind
}

}  // namespace

int32_t gemm_launch_mxs(const GemmParams& p, int grid_m, bool swiglu, bool once, hipStream_t st) {
  typedef MxsCfg C;
  GemmParams q = p;
  q.grid_n = (int)cdiv(p.N, C::BN);
  const int64_t tiles = (int64_t)grid_m * q.grid_n;
  if (tiles <= 0) return TK_OK;
  if (tiles > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_moe_gemm: grid too large");
  // a multiple of 8 workgroups (every XCD walks its share of the tiles), two per CU
  int64_t grid = (int64_t)busy_cu_count(p.idle_cus) * 2 / 8 * 8;
  grid = grid < 8 ? 8 : grid;
  grid = grid < cdiv(tiles, 8) * 8 ? grid : cdiv(tiles, 8) * 8;
  auto launch = [&](auto kern) -> int32_t {
    if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), C::LDS)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::NW * 64), C::LDS, st, q);
    return check_launch("moe_gemm_mxs_kernel");
  };
  if (once) return swiglu ? launch(moe_gemm_mxs_kernel<true, true>) : launch(moe_gemm_mxs_kernel<false, true>);
  return swiglu ? launch(moe_gemm_mxs_kernel<true, false>) : launch(moe_gemm_mxs_kernel<false, false>);
}

}  // namespace tk
