// Expert GEMM on tiled MXFP4 weights for more than a few rows per expert, bf16 or MXFP8 activations: tiles of 32 to 160 rows x 256 or 512
// columns with both operands staged by memory-to-LDS transfers.  Which tile a call gets, and why there: mxw_tile (gemm_limits.h).
//
//   * Four or eight waves, each all rows x 64 columns, two to a SIMD (four waves: two workgroups a CU).  Tiles of 512 columns halve what the rows cross from
//     L2.  160 rows (160 accumulators of a wave's 256 registers; a stage of 128 k moves 40 or 20 KiB of rows and 34 KiB of weights per 5120 / 2560
//     matrix cycles): an expert with 128 +- 11 rows is one tile, so its weights are read once.  The smaller ones bring fewer rows that are not there, and
//     have LDS for three stages of weights, which is what few rows per expert wait for (but 64 x 256, two workgroups a CU with two each), and up to 64 rows of three of
//     the rows too.
//   * Everything comes by `buffer_load ... lds`: no registers wait for memory, rows past the slice, columns past N and k past K are a matter of
//     the lanes' offsets (past the resource's range the hardware writes zeros).  Rings of two or three stages of rows and of weights run on
//     across the tiles of a persistent workgroup.
//   * bf16: e2m1 -> bf16 in registers in front of v_mfma_f32_32x32x16_bf16.  MXFP8: both operands as stored to
//     v_mfma_scale_f32_32x32x64_f8f6f4; a row's activation scales arrive sixteen blocks at a time, by transfers as well, and wait in LDS for four stages.
//   * What the next tile needs before its transfers (source rows) and in its epilogue (bias, gate weights, destinations) is fetched and parked in LDS one
//     stage before the rows' ring needs it.  No load into registers is on its way anywhere else: the compiler, which cannot count the transfers, waits
//     for all of them wherever such a load may be outstanding, and one that is requested in one stage and used in another may be in every
//     stage (128 experts of MXFP8 rows, layer, us: 9 rows 368 -> 293, 44 431 -> 395, 72 488 -> 444, 94 505 -> 479).  The epilogue's stores depend on nothing but the row fragments that hold
//     rows, so the wait in front of the next tile's first stage counts them and does not wait for them.
//
// What bounds the 160-row tile: the board's power in bf16 (fetching zeros instead of the weights, the operands then all zero, 558 -> 417 us; matrix pipe
// 68 % busy at 1.9 GHz), in MXFP8 no single part (360 us; without its multiplications 325, with the weights from L2 307, hardly any LDS reads 343, without
// the epilogue's arithmetic and stores 316): of a stage's 5500 cycles 2160 go into its multiplications, 1770 into waiting for transfers and the other waves,
// 870 into the epilogue's share and 370 into the next tile's words.  128 experts, K 2880, 4096 tokens, top-4, whole layer:
// bf16 861 -> 815 us, MXFP8 609 -> 563 us against the kernels that keep weights in registers with one wave per SIMD (moe_gemm_mxn, _mx8n, which
// serve what this one does not take).  The smaller ones: reading the weights (128 experts, 14 MXFP8 rows each, both GEMMs 305 us for 1.63 GB).  Measured
// and left out: transfers spread over the whole bf16 stage (576 against 558 us: the last ones are late); weights brought into L2 a stage ahead
// of their transfer (570 against 558, MXFP8 387 against 363 us); rings of four and six stages with 32 and 64 rows (no change); all four row fragments'
// epilogue whether they hold rows or not (128 x 512, 28 MXFP8 rows, both GEMMs 377 against 341 us).
#pragma once
#include "gemm_tiles.h"

namespace tk {
namespace {

// MFW_ row fragments, NW_ waves (each all rows x 64 columns), rings of ABUFS_ stages of rows and WBUFS_ of weights
template <bool MX8, int MFW_, int NW_, int ABUFS_, int WBUFS_>
struct MxwCfg {
  static constexpr int MFW = MFW_, NW = NW_;
  static constexpr int BM = MFW * 32, BN = NW * 64;
  static constexpr int ROW = MX8 ? 128 : 256;            // bytes of a row and stage (128 k)
  static constexpr int RPT = 1024 / ROW;                 // rows of a transfer
  static constexpr int AI = (BM / RPT + NW - 1) / NW;    // activation transfers of a wave and stage
  static constexpr bool HALF = BM / RPT % NW != 0;       // a wave's last one is half a transfer
  static_assert(!HALF || (BM / RPT) * 2 == (2 * AI - 1) * NW, "every wave has the same number of transfers");
  static constexpr int AWAVE = AI * 1024 - (HALF ? 512 : 0), ABYTES = AWAVE * NW;
  static constexpr int WWAVE = 4096 + 256, WBYTES = WWAVE * NW;  // a wave's two weight fragments: values, scales
  static constexpr int ABUFS = ABUFS_, WBUFS = WBUFS_;
  static constexpr int RINGS = ABUFS * ABYTES + WBUFS * WBYTES;
  static constexpr int SIDE = MX8 ? BM * 16 : 0;         // a row's activation scales of four stages
  static constexpr int RW = BM / NW, RAWI = (RW + 11) / 12;  // rows whose scales a wave fetches, its transfers for that (twelve rows each)
  static constexpr int RAW = MX8 ? RAWI * 256 * NW : 0;  // the scales as they arrive
  static constexpr int OPERANDS = (BN + 2 * BM) * 4;     // a tile's bias, gate weights, destination rows
  static constexpr bool LISTED = MFW == 5;               // the slice sizes and offsets wait in LDS: no registers are left for them
  static constexpr int LISTS = LISTED ? 2 * kDmaSlices * 4 : 0;
  static constexpr int LDS = RINGS + 2 * (SIDE + OPERANDS) + LISTS + RAW;
  static_assert(LDS <= 160 * 1024, "a CU's LDS");
};

// ONCE: the weights are fetched with the non-temporal hint (reads_once)
template <bool MX8, int MFW_, int NW_, int ABUFS_, int WBUFS_, bool SWIGLU, bool MXOUT, bool ONCE>
__global__ __launch_bounds__(NW_ * 64, 2) void moe_gemm_mxw_kernel(const GemmParams p) {
  typedef MxwCfg<MX8, MFW_, NW_, ABUFS_, WBUFS_> C;
  constexpr int MFW = C::MFW, AI = C::AI;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;
  const int nst = p.w_nst;
  const int KB = p.K * (MX8 ? 1 : 2);  // bytes of a row
  const uint32_t lds0 = lds_addr(lds);
  uint8_t* const side = lds + C::RINGS;
  float* const operands = reinterpret_cast<float*>(lds + C::RINGS + 2 * C::SIDE);

  // the tile list; its slice sizes and offsets in LDS between two tiles where they are LISTED (every wave stores the same words)
  int* const lists = reinterpret_cast<int*>(lds + C::RINGS + 2 * (C::SIDE + C::OPERANDS));
  typedef TileList<C::BM, C::BN> Tiles;
  Tiles list;
  int tile = list.init(p, lane, p.grid_n);
  const int t_step = list.t_step, t_end = list.t_end, f_beg = list.f_beg, f_len = list.f_len, s_beg = list.s_beg;
  if (tile >= t_end) return;
  Tile cur = list.locate(tile), nxt = cur;
  if constexpr (C::LISTED) {
#pragma unroll
    for (int c = 0; c < kSliceRegs; ++c) lists[c * 64 + lane] = list.sz[c], lists[kDmaSlices + c * 64 + lane] = list.so[c];
  }
  auto locate = [&](int i) __attribute__((always_inline)) -> Tile {
    if constexpr (!C::LISTED) return list.locate(i);
    Tiles t;
#pragma unroll
    for (int c = 0; c < kSliceRegs; ++c) t.sz[c] = lists[c * 64 + lane], t.so[c] = lists[kDmaSlices + c * 64 + lane];
    t.f_beg = f_beg, t.f_len = f_len, t.s_beg = s_beg, t.t_end = t_end, t.t_step = t_step, t.grid_n = p.grid_n;
    return t.locate(i);
  };
  const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(p.y, 0, (int)p.y_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ysrsrc = __builtin_amdgcn_make_buffer_rsrc(p.y_mx_scale, 0, MXOUT ? 0x7FFFFFFF : 0, 0x00020000);

  // ---- transfer side ------------------------------------------------------------------------------------------------------------------------------
  // activations: transfer i of this wave = rows (wave * AI + i) * RPT ..; lane -> row lane / (64 / RPT), its LDS position's piece swizzled by the row
  constexpr int LPR = 64 / C::RPT;  // lanes (16-byte pieces) of a row
  const buf_desc_t xdesc = make_buf_desc(p.x, p.x_bytes);
  buf_desc_t wdesc, sdesc;
  uint32_t a_off[AI];
  int raw_src[AI];                  // source rows of the next tile, on their way
  uint32_t raw_bias = 0, raw_gam = 0;
  int raw_dst = 0, raw_xs = 0;
  const uint32_t x_row = (uint32_t)(p.x_stride_m * (MX8 ? 1 : 2));
  auto row_of = [&](int i) __attribute__((always_inline)) -> int { return wave * (C::AWAVE / C::ROW) + i * C::RPT + lane / LPR; };
  auto piece_of = [&](int i) __attribute__((always_inline)) -> int {
    const int r = row_of(i);
    return MX8 ? ((lane & 7) ^ ((r >> 1) & 7)) : ((lane & 15) ^ (r & 15));
  };
  const int nfr = (p.N + 31) >> 5;
  const uint32_t f_val = (uint32_t)nst * 2048u, f_scale = (uint32_t)nst * 128u;  // bytes of a fragment
  const int scale_row = wave * C::RW + (lane < C::RW ? lane : C::RW - 1);  // the row whose activation scales this lane parks
  const uint32_t w_off = (uint32_t)lane * 16u, s_off = (uint32_t)h * f_scale + (uint32_t)lr * 4u;
  // what a tile needs from memory before its first transfers: source rows; and before its epilogue: bias, gate weights, destinations
  auto request = [&](const Tile& c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int row = c.off_m + row_of(i);
      const int sr = c.start_m + (row < c.eM ? row : c.eM - 1);
      raw_src[i] = p.gather ? p.gather[sr] : sr;
    }
    const int n = c.n_tile + tid < p.N ? c.n_tile + tid : p.N - 1;
    if (p.bias) {
      const int64_t i = (int64_t)c.expert * p.bias_stride_e + n;
      raw_bias = p.bias_is_f32 ? static_cast<const uint32_t*>(p.bias)[i] : (uint32_t)static_cast<const uint16_t*>(p.bias)[i];
    }
    int row = c.off_m + (tid < C::BM ? tid : C::BM - 1);
    const int sr = c.start_m + (row < c.eM ? row : c.eM - 1);
    if (p.gammas) raw_gam = p.gammas_is_f32 ? static_cast<const uint32_t*>(p.gammas)[sr] : (uint32_t)static_cast<const uint16_t*>(p.gammas)[sr];
    if (p.scatter) raw_dst = p.scatter[sr < p.scatter_len ? sr : p.scatter_len - 1];
    if constexpr (MX8) {
      row = c.off_m + scale_row;
      const int xr = c.start_m + (row < c.eM ? row : c.eM - 1);
      raw_xs = p.gather ? p.gather[xr] : xr;
    }
  };
  auto arrived = [&]() __attribute__((always_inline)) {  // (holds the uses of the requested words behind the wait in front of it)
#pragma unroll
    for (int i = 0; i < AI; ++i) asm volatile("" : "+v"(raw_src[i]));
    asm volatile("" : "+v"(raw_bias), "+v"(raw_gam), "+v"(raw_dst), "+v"(raw_xs));
  };
  auto park = [&](const Tile& c, int set) __attribute__((always_inline)) {
    float* const o = operands + set * (C::OPERANDS / 4);
    o[tid] = p.bias ? bits_f32(p.bias_is_f32 ? raw_bias : raw_bias << 16) : 0.f;
    if (tid < C::BM) {
      const int row = c.off_m + tid, sr = c.start_m + row;
      o[C::BN + tid] = p.gammas ? bits_f32(p.gammas_is_f32 ? raw_gam : raw_gam << 16) : 1.0f;
      int dst = sr;
      if (p.scatter) dst = sr < p.scatter_len ? raw_dst : -1;
      reinterpret_cast<int*>(o)[C::BN + C::BM + tid] = row < c.eM ? dst : -1;
    }
  };
  auto aim = [&](const Tile& c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AI; ++i)
      a_off[i] = c.off_m + row_of(i) < c.eM ? (uint32_t)raw_src[i] * x_row + (uint32_t)piece_of(i) * 16u : kOutOfRange;
  };
  auto aim_w = [&](const Tile& c) __attribute__((always_inline)) {
    // this wave's two fragments; past the last one nothing is in range (zeros: the columns are not stored)
    const int f0 = (c.n_tile >> 5) + wave * 2;
    const int nf = nfr - f0 < 0 ? 0 : nfr - f0 < 2 ? nfr - f0 : 2;
    wdesc = make_buf_desc(p.w + (int64_t)c.expert * p.w_stride_e + (int64_t)f0 * f_val, (uint32_t)nf * f_val);
    sdesc = make_buf_desc(p.w_scale + (int64_t)c.expert * p.ws_stride_e + (int64_t)f0 * f_scale, (uint32_t)nf * f_scale);
  };
  // transfers of stage s into a buffer: i of AI of the activations (k_end = bytes of a row), i of 5 of the weights; with nothing left to fetch
  // (k_end 0, !on) zeros, which nobody reads
  auto fetch_a = [&](int i, int s, uint32_t buf, int k_end) __attribute__((always_inline)) {
    const uint32_t at = s * C::ROW + piece_of(i) * 16 < k_end ? a_off[i] + (uint32_t)s * C::ROW : kOutOfRange, dst = lds0 + buf + wave * C::AWAVE + i * 1024;
    if (C::HALF && i == AI - 1)
      lds_dma16_lower(xdesc, dst, at);
    else
      lds_dma16(xdesc, dst, at);
  };
  auto fetch_w = [&](int i, int s, uint32_t buf, bool on) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + buf + wave * C::WWAVE;
    if (i < 4) {
      const int f = i >> 1, q = i & 1;
      lds_dma16<ONCE>(wdesc, dst + f * 2048 + q * 1024, (on ? (uint32_t)f * f_val + (uint32_t)s * 2048u + q * 1024u : kOutOfRange) + w_off);
    } else {
      lds_dma4<ONCE>(sdesc, dst + 4096, (on ? (uint32_t)s * 128u : kOutOfRange) + s_off);
    }
  };
  // Activation scales: sixteen blocks (four stages) of a row at a time.  They begin at any byte, so a transfer fetches the five words that hold them
  // (twelve rows a transfer), and a stage later the wave that fetched a row shifts them into place.  (Loads into registers, which the compiler knows of,
  // made it wait for everything outstanding in front of each stage's first operands.)
  const int kblocks = p.K >> 5;
  uint32_t xs_row = 0;
  const uint32_t xs_mis = MX8 ? (uint32_t)(reinterpret_cast<uintptr_t>(p.x_mx_scale) & 3) : 0u;
  const buf_desc_t xsdesc = make_buf_desc(p.x_mx_scale - xs_mis, MX8 ? (p.xs_bytes + xs_mis + 3u) & ~3u : 0u);
  const uint32_t raw0 = (uint32_t)(C::RINGS + 2 * (C::SIDE + C::OPERANDS) + C::LISTS + wave * C::RAWI * 256);
  auto scales_aim = [&]() __attribute__((always_inline)) { xs_row = (uint32_t)raw_xs * (uint32_t)p.xs_stride_m + xs_mis; };
  auto scales_request = [&](int g) __attribute__((always_inline)) {
    if constexpr (MX8) {
      const int r = (lane * 205) >> 10;  // lane / 5
#pragma unroll
      for (int i = 0; i < C::RAWI; ++i) {
        const uint32_t row = (uint32_t)__builtin_amdgcn_ds_bpermute((i * 12 + r) * 4, (int)xs_row);
        lds_dma4(xsdesc, lds0 + raw0 + i * 256, r < 12 ? ((row + (uint32_t)g * 16u) & ~3u) + (uint32_t)(lane - r * 5) * 4u : kOutOfRange);
      }
    }
  };
  auto scales_park = [&](int g, int set) __attribute__((always_inline)) {
    if constexpr (MX8) {
      if (lane < C::RW) {
        const int t = lane >= 12 ? 1 : 0;
        const uint32_t* raw = reinterpret_cast<const uint32_t*>(lds + raw0 + t * 256 + (lane - t * 12) * 20);
        uint32_t w[5];
#pragma unroll
        for (int d = 0; d < 5; ++d) w[d] = raw[d];
        u32x4_t o;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int in = kblocks - g * 16 - d * 4;  // blocks of this word inside the row; 2^0 behind its end
          const uint32_t keep = in >= 4 ? ~0u : in <= 0 ? 0u : (1u << (8 * in)) - 1u;
          o[d] = (__builtin_amdgcn_alignbyte(w[d + 1], w[d], xs_row) & keep) | (0x7F7F7F7Fu & ~keep);
        }
        *reinterpret_cast<u32x4_t*>(side + set * C::SIDE + scale_row * 16) = o;
      }
    }
  };

  // ---- the first tile: everything at once -----------------------------------------------------------------------------------------------------
  int set = 0, xset = 0;
  request(cur);
  arrived();
  park(cur, 0);
  aim(cur);
  if constexpr (MX8) scales_aim();
  scales_request(0);
  // the rings: activations one stage ahead, weights, which come from further away, WBUFS - 1
  constexpr uint32_t kW0 = C::ABUFS * C::ABYTES, kWEnd = C::RINGS;
  constexpr int AA = C::ABUFS - 1, WA = C::WBUFS - 1;
  uint32_t ab = 0, wb = kW0, wf_buf = kW0 + WA * C::WBYTES;  // buffers being read; the next one of the weights to fill
  aim_w(cur);
#pragma unroll
  for (int i = 0; i < 5; ++i) fetch_w(i, 0, kW0, true);
#pragma unroll
  for (int i = 0; i < AI; ++i) fetch_a(i, 0, 0, KB);
#pragma unroll
  for (int n = 1; n < (AA > WA ? AA : WA); ++n) {
#pragma unroll
    for (int i = 0; i < AI && n < AA; ++i) fetch_a(i, n, n * C::ABYTES, KB);
#pragma unroll
    for (int i = 0; i < 5 && n < WA; ++i) fetch_w(i, n, kW0 + n * C::WBYTES, true);
  }
  if constexpr (MX8) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(5 * WA + AI * AA) : "memory");  // (everything behind the scales)
    scales_park(0, 0);
  }
  bool more = true;
  int stored = 0;  // row fragments that the last epilogue has stored

  f32x16_t acc[2][MFW];
  // NJ = row fragments that hold rows (0: this wave has no columns)
  auto stages = [&](auto nj_c) __attribute__((always_inline)) {
    constexpr int NJ = decltype(nj_c)::value;
    for (int s = 0; s < nst; ++s) {
      // stage s has landed when only what was fetched behind it, the next stage's weights, is outstanding (and, in a tile's first stage, the
      // stores of the last epilogue); the buffers of stage s - 1 have been read
      constexpr int kBehind = AA == WA ? (AA - 1) * (AI + 5) : (WA - 1) * 5, kStores = MXOUT ? (SWIGLU ? 5 : 6) : 4;  // (stores of a fragment)
      static_assert(kBehind + MFW * kStores < 64, "what a wait can count");
      static_assert(WA <= AA + 1, "weights further ahead would let rows through that have not landed, and be aimed at the next tile before its words are there");
      if (s == 0) {
        static_for<0, MFW + 1>([&](auto n_c) __attribute__((always_inline)) {
          if (stored == decltype(n_c)::value) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kBehind + decltype(n_c)::value * kStores) : "memory");
        });
      } else {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kBehind) : "memory");
      }
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      int fs = s + AA, ws = s + WA;  // stages to fetch
      // the next tile: its words fetched and parked, a stage later its transfers begin.  (Requested a stage ahead the words are on their way across the
      // loop's other paths, and the compiler puts a wait for everything outstanding into every stage.)
      if (s == nst - AA - 1) {
        more = tile + t_step < t_end;
        if (more) {
          nxt = locate(tile + t_step);
          request(nxt);
          arrived();
          park(nxt, set ^ 1);
        } else {
          // (behind the last tile nothing is fetched: the words' wait, which is one for everything, cost products of one round 3 to 5 %, 64 slices of 8 bf16
          // rows, K 2880, N 512 21.2 us against 20.5, a layer of 1000 MXFP8 rows 102.5 against 99.9; the words get a value so that the old ones need no registers until here)
#pragma unroll
          for (int i = 0; i < AI; ++i) raw_src[i] = 0;
          raw_xs = 0;
        }
      } else if (s == nst - AA) {
        aim(nxt);
      }
      if (s == nst - WA) aim_w(nxt);
      if constexpr (MX8) {
        if (s == nst - 2) {
          scales_aim();
          scales_request(0);
        } else if (s == nst - 1) {
          scales_park(0, xset ^ 1);
        }
      }
      if constexpr (MX8) {
        if ((s & 3) == 1 && (s >> 2) + 1 <= ((nst - 1) >> 2)) scales_request((s >> 2) + 1);
        if ((s & 3) == 2 && (s >> 2) + 1 <= ((nst - 1) >> 2)) scales_park((s >> 2) + 1, xset ^ 1);
      }
      const bool w_on = more || ws < nst;
      ws = ws < nst ? ws : ws - nst;
      const int k_end = more || fs < nst ? KB : 0;
      fs = fs < nst ? fs : fs - nst;
      // (of the ring's buffers the one before the one being read)
      const uint32_t af_buf = AA == 1 ? ab ^ C::ABYTES : ab == 0 ? AA * C::ABYTES : ab - C::ABYTES;
      const uint8_t* a = lds + ab;
      const uint8_t* w = lds + wb + wave * C::WWAVE;
      auto fetch = [&](int i) __attribute__((always_inline)) {
        if (i < AI)
          fetch_a(i, fs, af_buf, k_end);
        else
          fetch_w(i - AI, ws, wf_buf, w_on);
      };
      if constexpr (NJ == 0) {
#pragma unroll
        for (int i = 0; i < AI + 5; ++i) fetch(i);
      } else {
        auto weights = [&](int f, int q) __attribute__((always_inline)) -> u32x4_t {
          return *reinterpret_cast<const u32x4_t*>(w + f * 2048 + q * 1024 + lane * 16);
        };
        // (a lane's two blocks of the stage)
        uint32_t sc[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) sc[f] = *reinterpret_cast<const uint16_t*>(w + 4096 + f * 128 + lr * 4 + 2 * h);
        if constexpr (MX8) {
          const uint8_t* xsc = side + xset * C::SIDE + lr * 16 + (s & 3) * 4 + 2 * h;
          const int sw = (lr >> 1) & 7;
          // two row fragments of a half stage ahead: activations, their scales; the second half's weights with its first one
          i32x8_t xf[3];
          uint32_t xs[3];
          u32x4_t wr[2][2];
          auto read = [&](auto i_c) __attribute__((always_inline)) {
            constexpr int i = decltype(i_c)::value, q = i / NJ, j = i % NJ;
            if constexpr (j == 0) wr[q][0] = weights(0, q), wr[q][1] = weights(1, q);
            const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(a + (j * 32 + lr) * 128 + (((q * 2 + h) ^ sw) * 16));
            const u32x4_t hi = *reinterpret_cast<const u32x4_t*>(a + (j * 32 + lr) * 128 + (((4 + q * 2 + h) ^ sw) * 16));
            xf[i % 3] = __builtin_bit_cast(i32x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            xs[i % 3] = *reinterpret_cast<const uint16_t*>(xsc + j * 512);
          };
          constexpr int NI = 2 * NJ;
          read(template_int<0>{});
          __builtin_amdgcn_sched_barrier(0);
          read(template_int<1>{});
          __builtin_amdgcn_sched_barrier(0);
          static_for<0, NI>([&](auto i_c) __attribute__((always_inline)) {
            constexpr int i = decltype(i_c)::value, q = i / NJ, j = i % NJ;
            if constexpr (i + 2 < NI) read(template_int<i + 2>{});
#pragma unroll
            for (int f = 0; f < 2; ++f) {
              // (an fp4 operand is the low four of the eight registers the builtin's type has; the others stay undefined)
              const i32x8_t wv = __builtin_bit_cast(i32x8_t, __builtin_shufflevector(wr[q][f], wr[q][f], 0, 1, 2, 3, -1, -1, -1, -1));
              acc[f][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, xf[i % 3], acc[f][j], 4 /* A: e2m1 */, 0 /* B: e4m3 */, q, (int)sc[f], q, (int)xs[i % 3]);
            }
            // (two transfers a step: late ones are waited for, four a step hold up the first multiplications; 94 rows of 128 experts, layer: 479 us,
            // 488 spread over the whole stage, 487 four a step)
            static_for<(2 * i < AI + 5 ? 2 * i : AI + 5), (2 * i + 2 < AI + 5 && i + 1 < NI ? 2 * i + 2 : AI + 5)>([&](auto t_c) __attribute__((always_inline)) { fetch(decltype(t_c)::value); });
            __builtin_amdgcn_sched_barrier(0);
          });
        } else {
          auto read = [&](auto i_c) __attribute__((always_inline)) -> bf16x8_t {
            constexpr int i = decltype(i_c)::value, t = i / NJ, j = i % NJ;
            return *reinterpret_cast<const bf16x8_t*>(a + (j * 32 + lr) * 256 + (((h * 8 + t) ^ (lr & 15)) * 16));
          };
          constexpr int NI = 8 * NJ, FPS = 3;  // transfers a step
          u32x4_t raw[2][2];
#pragma unroll
          for (int f = 0; f < 2; ++f) raw[f][0] = weights(f, 0), raw[f][1] = weights(f, 1);
          bf16x8_t xf[3], wf[2];
          xf[0] = read(template_int<0>{});
          xf[1] = read(template_int<1>{});
          __builtin_amdgcn_sched_barrier(0);
          // step t: lane half h supplies k = h * 64 + t * 8 .. + 7, which lie in MX block 2h + t / 4 of the stage
          static_for<0, NI>([&](auto i_c) __attribute__((always_inline)) {
            constexpr int i = decltype(i_c)::value, t = i / NJ, j = i % NJ;
            if constexpr (i + 2 < NI) xf[(i + 2) % 3] = read(template_int<(i + 2 < NI ? i + 2 : 0)>{});
#pragma unroll
            for (int f = 0; f < 2; ++f) {
              if constexpr (j == 0) wf[f] = dequant8(raw[f][t >> 2][t & 3], bits_f32(((sc[f] >> (8 * (t >> 2))) & 0xFFu) << 23));
              acc[f][j] = Frag<32>::mma(wf[f], xf[i % 3], acc[f][j]);
            }
            if constexpr (j == NJ - 1) {
              static_for<(t * FPS < AI + 5 ? t * FPS : AI + 5), (t * FPS + FPS < AI + 5 ? t * FPS + FPS : AI + 5)>([&](auto t_c) __attribute__((always_inline)) { fetch(decltype(t_c)::value); });
              __builtin_amdgcn_sched_barrier(0);
            }
          });
        }
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int j = 0; j < MFW; ++j) asm volatile("" : "+v"(acc[f][j]));
      }
      ab = AA == 1 ? ab ^ C::ABYTES : ab + C::ABYTES == kW0 ? 0 : ab + C::ABYTES;
      wb = wb + C::WBYTES == kWEnd ? kW0 : wb + C::WBYTES;
      wf_buf = wf_buf + C::WBYTES == kWEnd ? kW0 : wf_buf + C::WBYTES;
      if constexpr (MX8) xset ^= (s & 3) == 3 || s == nst - 1;
    }
  };

  while (true) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int j = 0; j < MFW; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[f][j][i] = 0.f;
    const int rows = cur.eM - cur.off_m < C::BM ? cur.eM - cur.off_m : C::BM;
    const int ncol0 = cur.n_tile + wave * 64;
    const int nj = ncol0 < p.N ? (rows + 31) >> 5 : 0;
    static_for<0, MFW + 1>([&](auto n_c) __attribute__((always_inline)) {
      if (nj == decltype(n_c)::value) stages(n_c);
    });
    const float* o = operands + set * (C::OPERANDS / 4);
    if constexpr (MXOUT)
      staged_mx_epilogue<MFW, 2, SWIGLU>(p, acc, yrsrc, ysrsrc, o, o + C::BN, reinterpret_cast<const int*>(o) + C::BN + C::BM, wave * 64, ncol0, lr, h, nj);
    else
      staged_epilogue<1, MFW, 2, 2, SWIGLU>(p, acc, yrsrc, o, o + C::BN, reinterpret_cast<const int*>(o) + C::BN + C::BM, wave * 64, ncol0, 0, lr, h, nj);
    if (!more) break;
    tile += t_step;
    cur = nxt;
    set ^= 1;
    stored = nj;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into this workgroup's LDS is left behind
}

template <bool MX8, int MFW, int NW, int ABUFS, int WBUFS>
int32_t launch_mxw(const GemmParams& p, bool swiglu, bool mx_out, hipStream_t st) {
  typedef MxwCfg<MX8, MFW, NW, ABUFS, WBUFS> C;
  constexpr int kPerCu = C::LDS <= 80 * 1024 && NW == 4 ? 2 : 1;  // workgroups of a CU
  static_assert(C::LDS * kPerCu <= 160 * 1024 && (NW == 8 || kPerCu == 2), "workgroups of a CU");
  static_assert(ABUFS + 1 <= 4, "a tile's events, the first of which comes ABUFS + 1 stages before its end, within the fewest stages of K that the kernel takes");
  GemmParams q = p;
  q.grid_n = (int)cdiv(p.N, C::BN);
  const int64_t tiles = (cdiv(p.M, C::BM) + (p.slice_sizes ? p.n_slices : 0)) * q.grid_n;  // at most
  if (tiles > 0x7FFFFFFF) return fail(TK_ERR_UNSUPPORTED, "tk_moe_gemm: grid too large");
  int64_t grid = (int64_t)busy_cu_count(p.idle_cus) * kPerCu / 8 * 8;  // every XCD walks its share of the tiles
  grid = grid < 8 ? 8 : grid;
  grid = grid < cdiv(tiles, 8) * 8 ? grid : cdiv(tiles, 8) * 8;
  auto launch = [&](auto kern) -> int32_t {
    if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), C::LDS)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::NW * 64), C::LDS, st, q);
    return check_launch("moe_gemm_mxw_kernel");
  };
  auto with = [&](auto once) -> int32_t {
    constexpr bool ONCE = decltype(once)::value;
    if constexpr (MX8) {
      if (mx_out) return swiglu ? launch(moe_gemm_mxw_kernel<true, MFW, NW, ABUFS, WBUFS, true, true, ONCE>) : launch(moe_gemm_mxw_kernel<true, MFW, NW, ABUFS, WBUFS, false, true, ONCE>);
    }
    return swiglu ? launch(moe_gemm_mxw_kernel<MX8, MFW, NW, ABUFS, WBUFS, true, false, ONCE>) : launch(moe_gemm_mxw_kernel<MX8, MFW, NW, ABUFS, WBUFS, false, false, ONCE>);
  };
  return reads_once(p.M, p.slice_sizes ? p.n_slices : 1, C::BM, p.N, p.K / 2) ? with(std::true_type{}) : with(std::false_type{});
}

}  // namespace
}  // namespace tk
