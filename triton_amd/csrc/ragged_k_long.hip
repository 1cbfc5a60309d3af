// Ragged-K GEMM (see ragged_k_gemm.hip) for aligned k-slow operands of slices long enough that the products, not the writing of y, take the time.
//
//   * A workgroup multiplies a T x T tile of one slice: 256 with eight waves of 128 x 64 (6 KiB of LDS reads for eight products, where a wave of 64 x 64
//     reads four for four, all that the LDS delivers), or 128 with four waves of 64 x 64 where those tiles would be few.
//   * A stage is 32 k of both operands, in the operands' own order by `buffer_load ... lds`; four stages are in LDS.  Its two steps of 16 k are read from LDS
//     (transposed, without bank conflicts) during the one before; the one barrier of a stage sits between them: behind it the next stage is
//     complete and this one has been read and is filled again.
//   * Workgroups are persistent and the ring runs on across tiles, so the first stages of a tile land during the epilogue of the one before, whose stores
//     nobody waits for until its fourth stage.
//   * Slices differ in length by factors: tiles go from the longest slice to the shortest, every XCD takes an eighth of each, and its workgroups walk
//     their list forth and back.  In a slice tiles run in bands of eight down, so that an XCD's 32 tiles share 12 operand columns instead of 15
//     (lines read past the L2 12.4 to 11.0 million a launch when the bands came in, 5 to 6 % of the time).
//
// What bounds it: 256 x 256, slices of thousands, the board's power (8 of 2048 k, 2880 x 5760 and 2880 x 2880: matrix pipe 69 % busy at 1.93 GHz, 1.0 PFLOP/s, where the vendor's
// library reaches 1.13 on a square product of 8192 of the same random numbers), slices of a hundred, the writing of y (128 of 128, 2880 x 5760: 29 % busy, 4.9 TB/s); 128 x 128, the lines that come to a CU (some 55 KB/us), and with few
// slices the longest.  Both products of a layer, us, the kernel for short slices / this one: 8 slices of 2048, d and f 2880 946 / 827; 32 of 512 1088 / 935; 128 of 128 1755 / 1623; 8 of
// 2048, d and f 512 140 / 85.
// Measured and left out: stores without the non-temporal hint (128 of 128, d and f 1440 421 -> 502), cleared accumulators in place of a first product on zero, whole rows of the tile an
// instruction as in the kernel for short slices (two barriers more per 32 rows; 128 of 128, d and f 2880 1628 -> 1656, rows that are no whole lines, 64 of 146, d 2016, f 1696 418 -> 416).
#include "ragged_k.h"

namespace tk {
namespace {

constexpr uint32_t kPastEnd = 0x80000000u;  // byte offset beyond every buffer resource here
constexpr int kRegs = kRaggedKLongSlices / 64;

// T x T tiles: 256 (eight waves of 128 x 64, one workgroup per CU) or 128 (four waves of 64 x 64, two per CU).
template <int T>
struct LongCfg {
  static constexpr int WM = 2, WN = T / 64, NW = WM * WN;
  static constexpr int MF = T / WM / 32, NF = 2;  // fragments of a wave
  static constexpr int KC = 32, BUFS = 4;         // k per stage, stages in LDS
  static constexpr int PITCH = T * 2;             // bytes of a k row
  static constexpr int OPERAND = KC * PITCH, STAGE = 2 * OPERAND, RING = BUFS * STAGE;
  static constexpr int OUT = 4096;                // bytes per wave for results on their way to whole lines
  static constexpr int LDS = RING + NW * OUT;
  static constexpr int TR = OPERAND / 1024 / NW;  // transfers of a wave, operand and stage
  static constexpr int PER_CU = T == 256 ? 1 : 2;
  static constexpr int STORES(int yt) { return yt == TK_F32 ? MF * NF * 4 : MF * 4; }
};
static_assert(LongCfg<256>::LDS == 160 * 1024 && LongCfg<128>::LDS == 80 * 1024, "one / two workgroups of a CU");

template <int DT, int YT, int T>
__global__ __launch_bounds__(LongCfg<T>::NW * 64, 2) void ragged_k_long_kernel(const RaggedKParams p) {
  typedef LongCfg<T> C;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;
  const int mw = wave % C::WM, nw = wave / C::WM;
  const uint32_t lds0 = lds_addr(lds);

  // ---- the slices, longest first: lane l of register c holds that of rank c * 64 + l ----------------------------------------
  int sz[kRegs], ao[kRegs], bo[kRegs], id[kRegs];
  {
    int* size_s = reinterpret_cast<int*>(lds);
    int* rank_s = size_s + kRaggedKLongSlices;
    int* id_s = rank_s + kRaggedKLongSlices;
    for (int e = tid; e < kRaggedKLongSlices; e += C::NW * 64) {
      size_s[e] = e < p.n_slices ? p.sizes[e] : -1;
      rank_s[e] = 0;
    }
    __syncthreads();
    // (each wave counts the longer ones, or as long and in front, among its share of the slices)
#pragma unroll
    for (int c = 0; c < kRegs; ++c) {
      const int e = c * 64 + lane, mine = size_s[e];
      int longer = 0;
      for (int o = wave; o < p.n_slices; o += C::NW) longer += size_s[o] > mine || (size_s[o] == mine && o < e) ? 1 : 0;
      if (e < p.n_slices) atomicAdd(&rank_s[e], longer);
    }
    __syncthreads();
    for (int e = tid; e < p.n_slices; e += C::NW * 64) id_s[rank_s[e]] = e;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kRegs; ++c) {
      const int r = c * 64 + lane < p.n_slices ? c * 64 + lane : 0;
      id[c] = id_s[r];
      sz[c] = size_s[id[c]];
      ao[c] = p.a_offs[id[c]], bo[c] = p.b_offs[id[c]];
    }
    // (here, and not at their first use, which the compiler cannot tell from later ones: a wait for them there would be a wait for the transfers)
#pragma unroll
    for (int c = 0; c < kRegs; ++c) asm volatile("" : "+v"(ao[c]), "+v"(bo[c]), "+v"(sz[c]), "+v"(id[c]));
    __syncthreads();
  }

  // ---- this workgroup's tiles: XCD b % 8 takes chunks of an eighth of a slice's tiles in turn; its workgroups walk them forth and back, so that
  // the sums of their lengths come out alike ---------------------------------------------------------------------------------
  const uint32_t per_e = (uint32_t)(p.tiles_m * p.tiles_n), total = per_e * (uint32_t)p.n_slices;
  const uint32_t q = (uint32_t)p.chunk, per_xcd = ((total + q - 1) / q + 7) / 8 * q;
  const uint32_t xcd = blockIdx.x & 7, i8 = blockIdx.x >> 3, wgs = gridDim.x >> 3;
  const uint32_t rounds = (per_xcd + wgs - 1) / wgs;
  struct Where {
    int id, ksz, a0, b0, m0, n0;
  };
  auto next = [&](uint32_t& r, Where& w) __attribute__((always_inline)) -> bool {
    for (; r < rounds; ++r) {
      const uint32_t l = r * wgs + (r & 1 ? wgs - 1 - i8 : i8), turn = l / q;
      const uint32_t pid = (turn * 8 + xcd) * q + (l - turn * q);
      if (l >= per_xcd || pid >= total) continue;
      const uint32_t rank = pid / per_e, in = pid - rank * per_e;
      // (bands of eight tiles down, in a band column by column, so that those in hand on an XCD share few operand columns)
      const uint32_t band = in / (8u * (uint32_t)p.tiles_n), left = (uint32_t)p.tiles_m - band * 8u, bh = left < 8u ? left : 8u;
      const uint32_t in_b = in - band * 8u * (uint32_t)p.tiles_n, tn = in_b / bh, tm = band * 8u + in_b - tn * bh;
#pragma unroll
      for (int c = 0; c < kRegs; ++c)
        if (kRegs == 1 || rank >> 6 == (uint32_t)c) {
          const int s = (int)(rank & 63);
          w.id = __builtin_amdgcn_readlane(id[c], s), w.ksz = __builtin_amdgcn_readlane(sz[c], s);
          w.a0 = __builtin_amdgcn_readlane(ao[c], s), w.b0 = __builtin_amdgcn_readlane(bo[c], s);
        }
      w.m0 = (int)tm * T, w.n0 = (int)tn * T;
      return true;
    }
    return false;
  };
  uint32_t cur_r = 0;
  Where cur;
  if (!next(cur_r, cur)) return;

  // ---- transfer side: the next stage to fetch -----------------------------------------------------------------------------------
  const buf_desc_t ra = make_buf_desc(p.a, p.a_bytes), rb = make_buf_desc(p.b, p.b_bytes);
  const uint32_t a_step = (uint32_t)p.a_stride_k * 2u, b_step = (uint32_t)p.b_stride_k * 2u;
  constexpr int PIECES = T / 8, ROWS = 64 / PIECES;  // 16-byte pieces of a k row, k rows of a transfer
  const int row0 = wave * C::TR * ROWS + lane / PIECES;  // (transfer i: + i * ROWS)
  uint32_t a_off[C::TR], b_off[C::TR];  // (past the edge: beyond the resource, and no sum of steps, which stays within 2 GiB, leads back)
  uint32_t f_r = cur_r;
  int f_left = 0;  // k of the tile aimed at that are still to be fetched
  auto aim = [&](const Where& w) __attribute__((always_inline)) {
    f_left = w.ksz;
#pragma unroll
    for (int i = 0; i < C::TR; ++i) {
      const int row = row0 + i * ROWS, piece = (lane % PIECES) ^ ((row & 3) * 4);
      const int m = w.m0 + piece * 8, n = w.n0 + piece * 8;
      a_off[i] = m < p.M ? (uint32_t)(w.a0 + row) * a_step + (uint32_t)m * 2u : kPastEnd;
      b_off[i] = n < p.N ? (uint32_t)(w.b0 + row) * b_step + (uint32_t)n * 2u : kPastEnd;
    }
  };
  auto issue = [&](uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C::TR; ++i) {
      const uint32_t dst = lds0 + buf + (uint32_t)(wave * C::TR + i) * 1024u;
      const bool in = row0 + i * ROWS < f_left;
      lds_dma16(ra, dst, in ? a_off[i] : kPastEnd);
      lds_dma16(rb, dst + C::OPERAND, in ? b_off[i] : kPastEnd);
      a_off[i] += a_step * C::KC, b_off[i] += b_step * C::KC;
    }
  };
  // behind the transfers of a stage: on to the next one, of this tile or of the next that has any (none left: zeros, read by nobody)
  auto advance = [&]() __attribute__((always_inline)) {
    f_left -= C::KC;
    while (f_left <= 0 && f_r < rounds) {
      Where w;
      ++f_r;
      if (!next(f_r, w)) break;
      aim(w);
    }
  };

  // ---- fragment reads (ragged_k_tr_kernel): a lane's row of four k, four columns; columns 32 j on are pieces 4 j on ---------------
  const int l16 = lane & 15, pp = ((lane >> 4) & 1) * 2 + ((l16 & 3) >> 1);
  const uint32_t rd0 = lds0 + (uint32_t)((h * 8 + (l16 >> 2)) * C::PITCH + (l16 & 1) * 8);
  uint32_t at_a[C::MF], at_b[C::NF];
#pragma unroll
  for (int j = 0; j < C::MF; ++j) at_a[j] = rd0 + (uint32_t)(((mw * C::MF * 4 + j * 4 + pp) ^ ((l16 >> 2) * 4)) * 16);
#pragma unroll
  for (int f = 0; f < C::NF; ++f) at_b[f] = rd0 + C::OPERAND + (uint32_t)(((nw * C::NF * 4 + f * 4 + pp) ^ ((l16 >> 2) * 4)) * 16);
  u32x4_t af[2][C::MF], bf[2][C::NF];
  auto read_a = [&](uint32_t buf, int s, int j) __attribute__((always_inline)) { return read_frag_tr(at_a[j] + (uint32_t)(s * 16 * C::PITCH) + buf, C::PITCH); };
  auto read_b = [&](uint32_t buf, int s, int f) __attribute__((always_inline)) { return read_frag_tr(at_b[f] + (uint32_t)(s * 16 * C::PITCH) + buf, C::PITCH); };

  f32x16_t acc[C::NF][C::MF];
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // half P of a stage: its products, while the operands of the next half (step 1 of the same stage, step 0 of the next) are read from `buf`
  // (FIRST: a tile's first, added to zero instead of to cleared registers)
  auto half = [&](auto p_c, auto first_c, uint32_t buf) __attribute__((always_inline)) {
    constexpr int P = decltype(p_c)::value;
    constexpr bool FIRST = decltype(first_c)::value;
#pragma unroll
    for (int f = 0; f < C::NF; ++f) bf[1 - P][f] = read_b(buf, 1 - P, f);
#pragma unroll
    for (int j = 0; j < C::MF; ++j) {
      af[1 - P][j] = read_a(buf, 1 - P, j);
#pragma unroll
      for (int f = 0; f < C::NF; ++f) acc[f][j] = mfma_k16<DT>(bf[P][f], af[P][j], FIRST ? zero : acc[f][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  uint32_t buf = 0;
  aim(cur);
  if (cur.ksz <= 0) {
    f_left = C::KC;  // (an empty tile: on to one that is not)
    advance();
  }
#pragma unroll
  for (int n = 0; n < C::BUFS; ++n) {
    issue(n * C::STAGE);
    advance();
  }
  constexpr int kPerStage = 2 * C::TR;
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((C::BUFS - 1) * kPerStage) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int f = 0; f < C::NF; ++f) bf[0][f] = read_b(0, 0, f);
#pragma unroll
  for (int j = 0; j < C::MF; ++j) af[0][j] = read_a(0, 0, j);

  // One stage.  NEWER = memory operations of this wave that may be outstanding when the next stage has landed: the two stages behind it and, in
  // the first three stages of a tile, the previous tile's stores, which were issued behind that stage's transfers.
  auto stage = [&](auto newer_c, auto first_c) __attribute__((always_inline)) {
    half(template_int<0>{}, first_c, buf);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(newer_c)::value) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this stage has been read
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(buf);
    buf = buf + C::STAGE == C::RING ? 0 : buf + C::STAGE;
    half(template_int<1>{}, std::false_type{}, buf);
    advance();
  };
  constexpr int kNewer = (C::BUFS - 2) * kPerStage;
  constexpr uint32_t ES = YT == TK_F32 ? 4 : 2;
  uint8_t* sp = lds + C::RING + wave * C::OUT;
  const uint32_t y_row = (uint32_t)p.y_stride_m * ES;
  bool stores = false;  // of the previous tile
  while (true) {
    const int nst = (cur.ksz + C::KC - 1) / C::KC;
    if (nst == 0) {
#pragma unroll
      for (int f = 0; f < C::NF; ++f)
#pragma unroll
        for (int j = 0; j < C::MF; ++j) acc[f][j] = zero;
    } else if (stores) {
      stage(template_int<kNewer + C::STORES(YT)>{}, std::true_type{});
      int s = 1;
      for (; s < (nst < C::BUFS - 1 ? nst : C::BUFS - 1); ++s) stage(template_int<kNewer + C::STORES(YT)>{}, std::false_type{});
      for (; s < nst; ++s) stage(template_int<kNewer>{}, std::false_type{});
    } else {
      stage(template_int<kNewer>{}, std::true_type{});
      for (int s = 1; s < nst; ++s) stage(template_int<kNewer>{}, std::false_type{});
    }
    stores = true;

    // ---- store: through LDS, so that an instruction writes eight whole 128-byte lines, with the non-temporal hint (32 bits: half lines as they are).
    // The resource ends behind row M - 1, so it drops rows past M by itself; columns past N start beyond it -------------------------------------------
    uint8_t* ye = p.y + (int64_t)cur.id * p.y_stride_e * ES;
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(ye, 0, p.y_bytes, 0x00020000);
    const int mb = cur.m0 + mw * C::MF * 32, nb = cur.n0 + nw * 64;
    if constexpr (YT == TK_F32) {
#pragma unroll
      for (int f = 0; f < C::NF; ++f)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int n = nb + f * 32 + u * 8 + h * 4;
          uint32_t off = n < p.N ? (uint32_t)(mb + lr) * y_row + (uint32_t)n * ES : kPastEnd;
#pragma unroll
          for (int j = 0; j < C::MF; ++j, off += 32u * y_row)
            __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{f32_bits(acc[f][j][4 * u]), f32_bits(acc[f][j][4 * u + 1]), f32_bits(acc[f][j][4 * u + 2]), f32_bits(acc[f][j][4 * u + 3])}, ry, off, 0, 0);
        }
    } else {
      const int n = nb + (lane & 7) * 8;
      uint32_t off = n < p.N ? (uint32_t)(mb + (lane >> 3)) * y_row + (uint32_t)n * ES : kPastEnd;
#pragma unroll
      for (int j = 0; j < C::MF; ++j) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        stage_out_rows<YT>(sp, 0, lane, acc[0][j], acc[1][j]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < 4; ++it, off += 8u * y_row)
          __builtin_amdgcn_raw_buffer_store_b128(staged_piece(sp, it * 8 + (lane >> 3), lane & 7), ry, off, 0, kNonTemporal);
      }
    }
    ++cur_r;
    if (!next(cur_r, cur)) break;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into this workgroup's LDS is left behind
}

template <int DT, int YT, int T>
int32_t launch_long(const RaggedKParams& p, hipStream_t st) {
  typedef LongCfg<T> C;
  RaggedKParams q = p;
  q.tiles_m = (int)cdiv(p.M, T), q.tiles_n = (int)cdiv(p.N, T);
  const int64_t per_e = (int64_t)q.tiles_m * q.tiles_n, total = per_e * p.n_slices;
  if (total > 0x7FFF0000) return fail(TK_ERR_UNSUPPORTED, "tk_ragged_k_gemm: grid too large");
  q.chunk = per_e >= 8 ? (int)(per_e / 8) : 1;
  int64_t grid = (int64_t)device_cu_count() * C::PER_CU / 8 * 8;
  const int64_t positions = cdiv(cdiv(total, q.chunk), 8) * 8 * q.chunk;
  grid = grid < 8 ? 8 : grid;
  grid = grid < positions ? grid : positions;
  auto kern = ragged_k_long_kernel<DT, YT, T>;
  if (const int32_t rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), C::LDS)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::NW * 64), C::LDS, st, q);
  return check_launch("ragged_k_long_kernel");
}

}  // namespace

int32_t ragged_k_launch_long(const RaggedKParams& p, int dtype, int tile, hipStream_t st) {
  auto with_y = [&](auto dt) -> int32_t {
    constexpr int DT = decltype(dt)::value;
    auto with_tile = [&](auto yt) -> int32_t {
      constexpr int YT = decltype(yt)::value;
      return tile == 256 ? launch_long<DT, YT, 256>(p, st) : launch_long<DT, YT, 128>(p, st);
    };
    return p.y_dtype == TK_BF16 ? with_tile(template_int<TK_BF16>{}) : p.y_dtype == TK_F16 ? with_tile(template_int<TK_F16>{}) : with_tile(template_int<TK_F32>{});
  };
  return dtype == TK_BF16 ? with_y(template_int<TK_BF16>{}) : with_y(template_int<TK_F16>{});
}

}  // namespace tk
