// Expert GEMM for full row blocks with both operands staged by memory-to-LDS transfers: bf16 / fp16 (strided, K-contiguous weights)
// and e4m3 (tiled weights), fp32 accumulation, the shared epilogue.
//
//   * A workgroup multiplies BM rows of one expert by BN columns: 256 x 256 with eight waves of 128 x 64 (one workgroup per CU),
//     128 x 128 with four waves of 64 x 64 (two per CU), or with 16-bit operands 320 x 256 or 320 x 128, eight waves of 160 x 64 or 160 x 32, for slices of
//     about 256 rows (dma_tile in gemm_limits.h, moe_gemm_dma_tall.hip).  Either way a SIMD holds two waves: while one waits for LDS or at the
//     barrier the other feeds the matrix pipe.
//   * A stage is 128 bytes of K of every row and column, i.e. whole cache lines: with 64-byte stages every line crossed from L2 to
//     the CU twice, 37 bytes per cycle for 18 useful ones.  The LDS holds two stages of activations and three of weights (which come
//     from further away; two beside 320 rows and 256 columns).  Every transfer is a `buffer_load ... lds` of 1 KiB per wave, eight rows of a line each: no registers, no VALU, no
//     LDS write instructions; gathered rows, rows past the slice, columns past N and k past K are a matter of the lanes'
//     offsets (past the resource's range the hardware writes zeros).
//   * Rows lie 128 bytes apart without padding (the transfer writes lane-contiguously); the 16-byte pieces of row r are stored at
//     piece ^ (r >> 1 & 7), so that sixteen rows read at one k occupy all banks once.  Tiled e4m3 blocks arrive in fragment order
//     and are read as they are.
//   * A stage is multiplied in four quarters; the operand fragments of a quarter are read from LDS during the one before.  The one
//     barrier of a stage sits in front of its last quarter: behind it the next stage is complete, this stage's buffers have been
//     read and are filled again.
//   * Workgroups are persistent and the ring runs on across tiles: the first stages of the next tile are on their way during the
//     last stages and the epilogue of this one.
//   * Short row blocks behind the last full round take half of the columns and twice the K a stage, so that all CUs have one and there are half
//     as many stages, each as long as its way from memory (bf16, us: 8 slices of about 1024 rows, K 2048, N 2048 79 -> 70, K 4096, N 4096 262 -> 240,
//     of about 512 rows 80 -> 73 and 156 -> 135; 16 of about 256, N 4096 85 to 95 -> 81).
//
// What bounds it: the board's power (a square bf16 product of 8192: matrix pipe 87 % busy at 1.58 GHz, 1390 TFLOP/s, 0.87 to 0.93 of what
// the vendor's library reaches on the same board), with shorter K also the epilogues (e4m3, K 4096: 12 % of the time; matrix pipe 67 % busy at 1.8
// GHz, K 14336: 77 % at 1.75), with a few rows per expert (128 x 128 tiles) the weight stream at 5.9 TB/s (5.3 without the
// non-temporal hint).  16384 routed rows
// of 8 experts in e4m3: K 4096, N 28672, swiglu 1840 -> 1590 us (2.42 PFLOP/s), K 14336, N 4096 850 -> 805 us; 4096 rows of 16
// experts in bf16, K 2048, about 256 rows each: a stage takes 1.9 to 2.4 us, twice its multiplications, and the CU's cache has about 90 lines of 128 bytes under way
// whatever is asked for ahead (weights two stages at a time into a ring of four: no change).  4096 rows of 16
// experts in bf16, K 2048: N 4096 231 -> 94 us, N 2048 133 -> 51 us (the kernels before: weights in registers with one wave
// per SIMD, and both operands through registers into LDS).
#pragma once
#include "gemm_tiles.h"

namespace tk {
namespace {

// 128 x 128 tiles (kDma128), 256 x 256 (kDma256), 320 x 256 and 320 x 128 (kDma320, kDma320Half; 16-bit operands)
enum { kDma128, kDma256, kDma320, kDma320Half };
template <int TILE>
struct DmaCfg {
  static constexpr int WM = 2, WN = TILE == kDma128 ? 2 : 4;                                       // waves along rows / columns
  static constexpr int MFW = TILE == kDma128 ? 2 : TILE == kDma256 ? 4 : 5, NFW = TILE == kDma320Half ? 1 : 2;  // fragments of a wave
  static constexpr int BM = WM * MFW * 32, BN = WN * NFW * 32;
  static constexpr int NW = WM * WN;
  static constexpr int ABYTES = BM * 128, BBYTES = BN * 128;
  static constexpr int ABUFS = 2, BBUFS = TILE == kDma320 ? 2 : 3;
  static constexpr int LDS = ABUFS * ABYTES + BBUFS * BBYTES;
  static constexpr int SBN = BN / 2;  // columns of a narrow tile
  static constexpr int AI = BM / 8 / NW, BI = BN / 8 / NW;  // transfers of a wave and stage
  static constexpr int PER_CU = TILE == kDma128 ? 2 : 1;    // workgroups
};
static_assert(DmaCfg<kDma256>::LDS == 160 * 1024 && DmaCfg<kDma128>::LDS == 80 * 1024 && DmaCfg<kDma320>::LDS <= 160 * 1024, "one / two workgroups of a CU");

// NARROW: short row blocks may be cut into narrow tiles (gemm_tiles.h).  ONCE: the weights are fetched with the non-temporal hint (reads_once).
// SMALL: all tiles are narrow ones, of row blocks half as high.
template <int WK, int TILE, bool SWIGLU, bool NARROW, bool ONCE, bool SMALL = false>
__device__ __forceinline__ void dma_gemm(const GemmParams& p) {
  typedef DmaCfg<TILE> C;
  constexpr bool F8 = WK == WK_FP8;
  constexpr int ES = F8 ? 1 : 2;
  constexpr int MFW = C::MFW, NFW = C::NFW;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mw = wave % C::WM, nw = wave / C::WM;
  const int lr = lane & 31, h = lane >> 5;
  const int KB = p.K * ES;                // bytes of a row
  const int nst = (KB + 127) >> 7;
  const uint32_t lds0 = lds_addr(lds);

  static_assert(NARROW || !SMALL, "small tiles are narrow ones");
  constexpr int LBM = SMALL ? C::BM / 2 : C::BM, LBN = SMALL ? C::SBN : C::BN;
  TileList<LBM, LBN, NARROW ? C::SBN : C::BN> tiles;
  int tile = tiles.init(p, lane, (p.N + LBN - 1) / LBN);
  auto locate = [&](int i) __attribute__((always_inline)) -> Tile {
    Tile t = tiles.locate(i);
    if (SMALL) t.narrow = true;
    return t;
  };
  const int t_step = tiles.t_step, t_end = tiles.t_end;
  if (tile >= t_end) return;

  // ---- transfer side ------------------------------------------------------------------------------------------------------------------------------
  // transfer i of an operand: rows i * 8 .. + 7, lane -> row lane / 8, LDS position lane % 8, i.e. piece (lane % 8) ^ (row >> 1 & 7);
  // with eight rows a transfer, row >> 1 & 7 = (i & 1) * 4 + (lane >> 4)
  // (pc0, pc1: of a wave's transfers of even and odd index, which start at an even index or, of activations, at wave * AI)
  const int pc0 = (lane & 7) ^ (lane >> 4), pc1 = pc0 ^ 4;
  const int pa0 = C::AI % 2 ? pc0 ^ ((wave & 1) << 2) : pc0, pa1 = pa0 ^ 4;
  const buf_desc_t xdesc = make_buf_desc(p.x, p.x_bytes);
  buf_desc_t wdesc;
  uint32_t a_off[C::AI], b_off[C::BI];
  const uint32_t x_row = (uint32_t)(p.x_stride_m * ES);
  static_assert(C::BI % 2 == 0 && (C::AI % 2 == 0 || !NARROW), "a transfer's parity is that of its index in the wave");
  // A narrow tile's stage is twice as long: the first half of the waves fetches its first 128 bytes of K, for half of the rows and columns that the
  // buffers have room for, the others the second.
  int f_step = 128, f_kh = 0;  // bytes of K of a stage, and where this wave's transfers begin in it
  auto aim = [&](const Tile& c) __attribute__((always_inline)) {
    const bool nar = NARROW && c.narrow;
    if constexpr (NARROW) {
      f_step = nar ? 256 : 128;
      f_kh = nar ? wave / (C::NW / 2) * 128 : 0;
    }
    const int w_in = nar ? wave % (C::NW / 2) : wave;
#pragma unroll
    for (int i = 0; i < C::AI; ++i) {
      const int row = c.off_m + (w_in * C::AI + i) * 8 + (lane >> 3);
      const int sr = c.start_m + (row < c.eM ? row : c.eM - 1);
      const uint32_t src = p.gather ? (uint32_t)p.gather[sr] : (uint32_t)sr;
      a_off[i] = row < c.eM ? src * x_row + (uint32_t)((i & 1) ? pa1 : pa0) * 16u : kOutOfRange;
    }
    const uint8_t* w = p.w + (int64_t)c.expert * p.w_stride_e;
    if constexpr (F8) {
      const int f0 = c.n_tile >> 5, nfr = (p.N + 31) >> 5, nf = C::BN / 32;
      const uint32_t fsz = (uint32_t)p.w_nst * 8192u;  // bytes of a column fragment
      wdesc = make_buf_desc(w + (int64_t)f0 * fsz, (uint32_t)(nfr - f0 < nf ? nfr - f0 : nf) * fsz);
#pragma unroll
      for (int i = 0; i < C::BI; ++i) {
        const int id = w_in * C::BI + i;  // KiB id % 4 of fragment id / 4's block
        b_off[i] = (uint32_t)(id >> 2) * fsz + (uint32_t)(id & 3) * 1024u + (uint32_t)lane * 16u;
      }
    } else {
      const int bn = nar ? C::SBN : C::BN, cols = p.N - c.n_tile < bn ? p.N - c.n_tile : bn;
      wdesc = make_buf_desc(w + (int64_t)c.n_tile * p.w_stride_n, (uint32_t)(cols - 1) * (uint32_t)p.w_stride_n + (uint32_t)KB);
#pragma unroll
      for (int i = 0; i < C::BI; ++i) {
        const int n = (w_in * C::BI + i) * 8 + (lane >> 3);
        b_off[i] = n < cols ? (uint32_t)n * (uint32_t)p.w_stride_n + (uint32_t)((i & 1) ? pc1 : pc0) * 16u : kOutOfRange;
      }
    }
  };
  // transfer i of this wave for the stage at byte kb of K of the tile aimed at (none left: zeros into a buffer that nobody reads)
  auto fetch_a = [&](int i, int kb, uint32_t buf, bool more) __attribute__((always_inline)) {
    kb += f_kh;
    const bool in = more && kb + ((i & 1) ? pa1 : pa0) * 16 < KB;
    lds_dma16(xdesc, lds0 + buf + (wave * C::AI + i) * 1024, in ? a_off[i] + (uint32_t)kb : kOutOfRange);
  };
  auto fetch_b = [&](int i, int kb, uint32_t buf, bool more) __attribute__((always_inline)) {
    kb += f_kh;
    const bool in = more && (F8 ? !NARROW || kb < KB : kb + ((i & 1) ? pc1 : pc0) * 16 < KB);  // (blocks of tiled weights are padded with zeros)
    lds_dma16<ONCE>(wdesc, lds0 + buf + (wave * C::BI + i) * 1024, in ? b_off[i] + (uint32_t)kb * (F8 ? 32u : 1u) : kOutOfRange);
  };

  // ---- LDS read side ----------------------------------------------------------------------------------------------------------------------------
  // 16-bit: step t of four, the lane's piece 2t + h;  e4m3: step u of two, the lane's pieces 4u + 2h + {0, 1} (32 consecutive k)
  const int sw = (lr >> 1) & 7;
  uint32_t pos[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) pos[t] = (uint32_t)(((F8 ? (t >> 1) * 4 + 2 * h + (t & 1) : 2 * t + h) ^ sw) * 16 + lr * 128);
  auto ld = [&](uint32_t at) __attribute__((always_inline)) -> u32x4_t { return *reinterpret_cast<const u32x4_t*>(lds + at); };
  auto read_a = [&](uint32_t buf, int j, int t) __attribute__((always_inline)) -> u32x4_t {
    return ld(buf + (uint32_t)(mw * 4096) + pos[t] + j * (C::WM * 4096));
  };
  auto read_b = [&](uint32_t buf, int f, int t) __attribute__((always_inline)) -> u32x4_t {
    return F8 ? ld(buf + (uint32_t)(nw * NFW * 4096) + (uint32_t)lane * 16u + f * 4096 + t * 1024) : ld(buf + (uint32_t)(nw * NFW * 4096) + pos[t] + f * 4096);
  };

  // ---- the rings: one cursor, two stages ahead of the multiplication --------------------------------------------------------------------------
  constexpr uint32_t kAEnd = C::ABUFS * C::ABYTES, kBEnd = kAEnd + C::BBUFS * C::BBYTES;
  Tile cur = locate(tile);
  aim(cur);
  uint32_t aw = 0, bw = kAEnd;  // buffers the next transfers fill
  int fs = 0;                   // where the next stage to fetch begins
  bool more = true;
  int f_tile = tile;
  auto advance = [&]() __attribute__((always_inline)) {
    aw = aw + C::ABYTES == kAEnd ? 0 : aw + C::ABYTES;
    bw = bw + C::BBYTES == kBEnd ? kAEnd : bw + C::BBYTES;
    if ((fs += f_step) >= KB) {
      fs = 0;
      f_tile += t_step;
      more = more && f_tile < t_end;
      if (more) aim(locate(f_tile));
    }
  };

  f32x16_t acc[NFW][MFW];
  auto mma16 = [&](u32x4_t w, u32x4_t x, f32x16_t c) __attribute__((always_inline)) -> f32x16_t {
    if constexpr (WK == WK_F16)
      return Frag<32>::mma_f16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), c);
    else
      return Frag<32>::mma(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), c);
  };
  auto both = [&](u32x4_t lo, u32x4_t hi) __attribute__((always_inline)) -> i32x8_t {
    return __builtin_bit_cast(i32x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Operand registers of the even and the odd quarters.  16-bit: quarter t multiplies step t, all row fragments.  e4m3: quarters 2u and
  // 2u + 1 multiply the lower and the upper half of the row fragments of step u; the weights of a step live in w8[u].
  u32x4_t ar[2][F8 ? 1 : MFW], wr[2][F8 ? 1 : NFW];
  i32x8_t a8[2][F8 ? MFW / 2 : 1], w8[2][F8 ? NFW : 1];
  // quarter Q of the stage at (abuf, bbuf), while the operands of the next quarter are read: of the same stage, or for Q = 3 of the next
  // (NJ row fragments if that is not 0, else those of the wave's MFW that hold rows)
  auto quarter = [&](auto nj_c, auto q_c, int jc, uint32_t abuf, uint32_t bbuf) __attribute__((always_inline)) {
    constexpr int NJ = decltype(nj_c)::value, JN = NJ ? NJ : MFW;
    constexpr bool FULL = NJ != 0;
    constexpr int Q = decltype(q_c)::value, QN = (Q + 1) & 3, P = Q & 1;
    // A wave's transfers are spread over the stage (the CU takes one per sixteen cycles or so; all eight behind the barrier held up
    // its first multiplications): activations, which the next barrier waits for, in quarter 3, weights in quarters 0 and 1.
    // (With two stages of weights these wait for the barrier as well, and go first: they come from further away.)
    constexpr int QB = C::BBUFS == 2 ? (Q == 3 ? C::BI : 0) : Q < 2 ? C::BI / 2 : 0, QT = QB + (Q == 3 ? C::AI : 0);
    auto transfer = [&](int k, int of) __attribute__((always_inline)) {
#pragma unroll
      for (int i = k * QT / of; i < (k + 1) * QT / of; ++i) {
        if (i < QB)
          fetch_b(C::BBUFS == 2 ? i : Q * QB + i, fs, bw, more);
        else
          fetch_a(i - QB, fs, aw, more);
      }
    };
    if constexpr (!F8) {
#pragma unroll
      for (int f = 0; f < NFW; ++f) wr[1 - P][f] = read_b(bbuf, f, QN);
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        ar[1 - P][j] = read_a(abuf, j, QN);
        if (FULL || j < jc) {
#pragma unroll
          for (int f = 0; f < NFW; ++f) acc[f][j] = mma16(wr[P][f], ar[P][j], acc[f][j]);
        }
        if constexpr (MFW % 2 == 0) {
          if (j % (MFW / 2) == MFW / 2 - 1) transfer(j / (MFW / 2), 2);
        } else {
          transfer(j, JN);
        }
        if constexpr (FULL) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      constexpr int U = Q >> 1, UN = QN >> 1, HJ = MFW / 2;
#pragma unroll
      for (int j = 0; j < HJ; ++j) {
        a8[1 - P][j] = both(read_a(abuf, (1 - P) * HJ + j, 2 * UN), read_a(abuf, (1 - P) * HJ + j, 2 * UN + 1));
        if constexpr (P == 1) {  // the weights of the next step
#pragma unroll
          for (int f = j * NFW / HJ; f < (j + 1) * NFW / HJ; ++f) w8[1 - U][f] = both(read_b(bbuf, f, 2 * UN), read_b(bbuf, f, 2 * UN + 1));
        }
        if (FULL || P * HJ + j < jc) {
#pragma unroll
          for (int f = 0; f < NFW; ++f)
            acc[f][P * HJ + j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8[U][f], a8[P][j], acc[f][P * HJ + j], 0, 0, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
        }
#pragma unroll
        for (int k = 0; k < 2 / HJ; ++k) transfer(HJ == 2 ? j : k, 2);
        if constexpr (FULL) {
          // (an empty use of the results: the compiler otherwise sinks the multiplications to the end of the loop)
#pragma unroll
          for (int f = 0; f < NFW; ++f) asm volatile("" : "+v"(acc[f][P * HJ + j]));
        }
        if constexpr (FULL) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // stages 0 and 1 of both operands: as the loop finds them in front of its quarter 0
#pragma unroll
  for (int n = 0; n < 2; ++n) {
#pragma unroll
    for (int i = 0; i < C::BI; ++i) fetch_b(i, fs, bw, more);
#pragma unroll
    for (int i = 0; i < C::AI; ++i) fetch_a(i, fs, aw, more);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::AI + C::BI) : "memory");
  barrier();
  uint32_t ab = 0, bb = kAEnd;
  // the operands of a tile's first quarter (read again behind an epilogue, which needs the registers)
  auto prime = [&]() __attribute__((always_inline)) {
    if constexpr (!F8) {
#pragma unroll
      for (int f = 0; f < NFW; ++f) wr[0][f] = read_b(bb, f, 0);
#pragma unroll
      for (int j = 0; j < MFW; ++j) ar[0][j] = read_a(ab, j, 0);
    } else {
#pragma unroll
      for (int f = 0; f < NFW; ++f) w8[0][f] = both(read_b(bb, f, 0), read_b(bb, f, 1));
#pragma unroll
      for (int j = 0; j < MFW / 2; ++j) a8[0][j] = both(read_a(ab, j, 0), read_a(ab, j, 1));
    }
  };
  // A narrow tile, BM / 2 rows by SBN columns, 32 columns a wave: what takes its time is not the multiplications but a stage's way from memory,
  // and a stage is as many bytes as a full tile's.
  auto narrow_tile = [&]() __attribute__((always_inline)) {
    constexpr int MH = MFW / 2;
    f32x16_t part[1][MH];
#pragma unroll
    for (int j = 0; j < MH; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) part[0][j][i] = 0.f;
    const int jn = __builtin_amdgcn_readfirstlane((((cur.eM - cur.off_m + 31) >> 5) - mw + C::WM - 1) / C::WM);
#pragma unroll 1
    for (int s = 0; s < (nst + 1) >> 1; ++s) {
#pragma unroll
      for (int i = 0; i < C::BI; ++i) fetch_b(i, fs, bw, more);
      if (jn > 0) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          const uint32_t a0 = ab + kh * (C::ABYTES / 2) + (uint32_t)(mw * 4096), b0 = bb + kh * (C::BBYTES / 2) + (uint32_t)(nw * 4096);
          u32x4_t w[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) w[t] = F8 ? ld(b0 + (uint32_t)lane * 16u + t * 1024) : ld(b0 + pos[t]);
#pragma unroll
          for (int j = 0; j < MH; ++j) {
            if (j >= jn) break;
            u32x4_t x[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) x[t] = ld(a0 + pos[t] + j * (C::WM * 4096));
            if constexpr (F8) {
#pragma unroll
              for (int u = 0; u < 2; ++u)
                part[0][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(both(w[2 * u], w[2 * u + 1]), both(x[2 * u], x[2 * u + 1]), part[0][j], 0, 0, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
            } else {
#pragma unroll
              for (int t = 0; t < 4; ++t) part[0][j] = mma16(w[t], x[t], part[0][j]);
            }
          }
        }
      }
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::BI) : "memory");
      barrier();
#pragma unroll
      for (int i = 0; i < C::AI; ++i) fetch_a(i, fs, aw, more);
      ab = ab + C::ABYTES == kAEnd ? 0 : ab + C::ABYTES;
      bb = bb + C::BBYTES == kBEnd ? kAEnd : bb + C::BBYTES;
      advance();
    }
    gemm_epilogue<32, C::WM, MH, 1, SWIGLU, WK == WK_F16>(p, part, cur.expert, cur.off_m, cur.start_m, cur.eM, cur.n_tile + nw * 32, cur.n_tile + C::SBN <= p.N, mw, lr, h);
  };
  while (true) {
    if (NARROW && cur.narrow) {
      narrow_tile();
      tile += t_step;
      if (tile >= t_end) break;
      cur = locate(tile);
      continue;
    }
    if constexpr (!SMALL) {
      prime();
#pragma unroll
      for (int f = 0; f < NFW; ++f)
#pragma unroll
        for (int j = 0; j < MFW; ++j)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[f][j][i] = 0.f;
      const int rows = cur.eM - cur.off_m < C::BM ? cur.eM - cur.off_m : C::BM;
      const int jc = __builtin_amdgcn_readfirstlane((((rows + 31) >> 5) - mw + C::WM - 1) / C::WM);  // this wave's row fragments (j * WM + mw) that hold rows
      auto stages = [&](auto nj_c) __attribute__((always_inline)) {
        for (int s = 0; s < nst; ++s) {
          quarter(nj_c, template_int<0>{}, jc, ab, bb);
          quarter(nj_c, template_int<1>{}, jc, ab, bb);
          quarter(nj_c, template_int<2>{}, jc, ab, bb);
          // the next stage has landed (this wave's part) when only the transfers of quarters 0 and 1 are outstanding
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::BBUFS == 2 ? 0 : C::BI) : "memory");
          barrier();
          ab = ab + C::ABYTES == kAEnd ? 0 : ab + C::ABYTES;
          bb = bb + C::BBYTES == kBEnd ? kAEnd : bb + C::BBYTES;
          quarter(nj_c, template_int<3>{}, jc, ab, bb);
          // (the one branch of a stage stands at its end: with one in between, the compiler moves the multiplications in front of it
          // down behind it, and their operands pile up)
          advance();
        }
      };
      if (jc >= MFW)
        stages(template_int<MFW>{});
      else if (MFW == 5 && jc == 4)
        stages(template_int<MFW == 5 ? 4 : 0>{});
      else
        stages(template_int<0>{});
      gemm_epilogue<32, C::WM, MFW, NFW, SWIGLU, WK == WK_F16>(p, acc, cur.expert, cur.off_m, cur.start_m, cur.eM, cur.n_tile + nw * NFW * 32,
                                                               cur.n_tile + C::BN <= p.N, mw, lr, h);
      tile += t_step;
      if (tile >= t_end) break;
      cur = locate(tile);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into this workgroup's LDS is left behind
}

template <int WK, int TILE, bool SWIGLU, bool NARROW, bool ONCE, bool SMALL = false>
__global__ __launch_bounds__(DmaCfg<TILE>::NW * 64, 2) void moe_gemm_dma_kernel(const GemmParams p) {
  dma_gemm<WK, TILE, SWIGLU, NARROW, ONCE, SMALL>(p);
}

// Workgroups of a launch over `tiles` tiles at most: a multiple of 8 (every XCD walks its share of the tiles), `per_cu` per CU at most.
inline unsigned dma_grid(const GemmParams& p, int per_cu, int64_t tiles) {
  int64_t grid = (int64_t)busy_cu_count(p.idle_cus) * per_cu / 8 * 8;
  grid = grid < 8 ? 8 : grid;
  return (unsigned)(grid < cdiv(tiles, 8) * 8 ? grid : cdiv(tiles, 8) * 8);
}

}  // namespace
}  // namespace tk
