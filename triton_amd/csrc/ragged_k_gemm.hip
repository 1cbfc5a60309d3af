// GEMM whose REDUCTION dimension is ragged (the expert weight gradient of a MoE layer):
//   y[e, m, n] = sum over k < sizes[e] of a[m, a_offs[e] + k] * b[b_offs[e] + k, n]
// Follows tk/matmul.py:376-384 (`b_ragged_metadata` selects ragged_dimension "K", one output per slice),
// tk/matmul_details/_matmul.py:252-272 (a slice's k range comes from the slice offsets of BOTH operands, its length
// from the slice sizes) and the torch statement of it in tk/matmul.py:852-875.
//
// In the weight-gradient use a = x^T [hidden, rows] and b = dy [rows, n] are both stored with the reduction index as
// the SLOW dimension, while an MFMA lane wants 8 consecutive k of one row.  The transposition happens between the
// global load and LDS: a thread fetches four k rows of the same eight m (four 16-byte loads, coalesced along m),
// interleaves them in registers and writes eight 8-byte pieces [m][k..k+3]; the MFMA operands are then plain
// 16-byte LDS reads.  An operand stored k-contiguous skips the interleave.  Anything that is not 16-byte aligned or
// hangs over an edge takes an element-wise path with zero fill (k past the slice MUST read as zero: the neighbouring
// rows belong to another expert).
//
// The problem is bound by writing y (n_slices * M * N outputs from short reductions), not by the MFMAs: at 128
// experts x 2880 x 5760 from 256 rows each the output is 4.2 GB against 1.1 TFLOP.
#include <algorithm>
#include <type_traits>

#include "ragged_k.h"

namespace tk {
namespace {

constexpr int kTile = 128;  // output tile edge (rows and columns)
constexpr int kKC = 32;     // k per pipeline stage
constexpr int kRing = 3;   // stages of global loads in flight per thread
constexpr int kPitch = kKC * 2 + 16;  // bytes per LDS row: 32 k + a pad that keeps 16-byte alignment and spreads banks

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for_n(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for_n<N, I + 1>(f);
  }
}
template <class F>
__device__ __forceinline__ void static_for_ring(F&& f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  static_assert(kRing == 3, "static_for_ring lists the slots");
}

// Any layout and alignment (the aligned k-slow pair runs ragged_k_tr_kernel below).
template <int DT>
__global__ __launch_bounds__(256) void ragged_k_gemm_kernel(const RaggedKParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][kTile * kPitch];  // [buffer][operand][row][k]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;
  const int mw = wave & 1, nw = wave >> 1;  // the wave's 64 x 64 quadrant

  // workgroups go round-robin to the 8 XCDs; renumber so that consecutive tiles, which share a slice's operand rows,
  // run on one XCD and find them in its L2
  int pid;
  {
    const int total = gridDim.x, per = total / 8, extra = total % 8;
    const int grp = blockIdx.x % 8, local = blockIdx.x / 8;
    pid = grp * per + (grp < extra ? grp : extra) + local;
  }
  const int tn = pid % p.tiles_n;
  pid /= p.tiles_n;
  const int tm = pid % p.tiles_m;
  const int e = pid / p.tiles_m;
  const int ksz = p.sizes[e];
  const int a_k0 = p.a_offs[e], b_k0 = p.b_offs[e];
  const int m0 = tm * kTile, n0 = tn * kTile;

  // ---- this thread's piece of a stage: threads 0..127 stage operand a, 128..255 operand b ----
  const bool is_b = tid >= 128;
  const int t7 = tid & 127;
  const uint8_t* base = is_b ? p.b : p.a;
  const int64_t stride_r = is_b ? p.b_stride_n : p.a_stride_m;
  const int64_t stride_k = is_b ? p.b_stride_k : p.a_stride_k;
  const int k_first = is_b ? b_k0 : a_k0;
  const int r0 = is_b ? n0 : m0;
  const int rows_total = is_b ? p.N : p.M;
  const bool vec_ok = (is_b ? p.b_vec : p.a_vec) != 0;
  const bool k_slow = stride_r == 1;
  // k-slow: piece = 4 k rows (kq*4 ..) x 8 rows (rb*8 ..);  k-contiguous: piece = one row x 32 k
  // kq runs fastest over the lanes: the eight lanes of one row block write 64 contiguous bytes of an LDS row, and row
  // blocks (8 rows = 640 bytes apart) alternate between two bank phases, so an LDS write sees a 2-way conflict at most
  // (with the row block fastest, sixteen lanes would share each bank); a load instruction still covers whole 128-byte
  // lines (8 lanes x 16 bytes along m)
  const int rb = t7 >> 3, kq = t7 & 7;
  // staged registers, a ring of kRing stages: k-slow 4 x uint4 = [k][8 rows]; k-contiguous 4 x uint4 = 32 k of one row
  uint32_t ring[kRing][16];
  uint8_t* my_lds0 = &lds[0][is_b ? 1 : 0][0];

  auto load_elem = [&](int64_t r, int64_t k) __attribute__((always_inline)) -> uint32_t {
    return *reinterpret_cast<const uint16_t*>(base + ((r0 + r) * stride_r + (k_first + k) * stride_k) * 2);
  };
  auto load_stage = [&](auto slot_c, int kc) __attribute__((always_inline)) {
    uint32_t(&pr)[16] = ring[decltype(slot_c)::value];
    if (k_slow) {
      const int rr = rb * 8;
      const bool full_rows = r0 + rr + 8 <= rows_total;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = kc + kq * 4 + q;
        if (k < ksz && vec_ok && full_rows) {
          const uint4 v = *reinterpret_cast<const uint4*>(base + ((int64_t)(r0 + rr) + (int64_t)(k_first + k) * stride_k) * 2);
          pr[4 * q + 0] = v.x;
          pr[4 * q + 1] = v.y;
          pr[4 * q + 2] = v.z;
          pr[4 * q + 3] = v.w;
        } else {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            uint32_t lo = 0, hi = 0;
            if (k < ksz) {
              if (r0 + rr + 2 * d < rows_total) lo = load_elem(rr + 2 * d, k);
              if (r0 + rr + 2 * d + 1 < rows_total) hi = load_elem(rr + 2 * d + 1, k);
            }
            pr[4 * q + d] = lo | (hi << 16);
          }
        }
      }
    } else {
      const int r = t7;
      const bool row_ok = r0 + r < rows_total;
      const uint8_t* rowp = base + ((int64_t)(r0 + r) * stride_r + (int64_t)k_first * stride_k) * 2;
      // 16-byte loads need k contiguous, the row start 16-byte aligned (the slice offset decides) and a full piece
      const bool can_vec = vec_ok && stride_k == 1 && row_ok && ((reinterpret_cast<uintptr_t>(rowp) & 15) == 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = kc + q * 8;
        if (can_vec && k + 8 <= ksz) {
          const uint4 v = *reinterpret_cast<const uint4*>(rowp + (int64_t)k * 2);
          pr[4 * q + 0] = v.x;
          pr[4 * q + 1] = v.y;
          pr[4 * q + 2] = v.z;
          pr[4 * q + 3] = v.w;
        } else {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            uint32_t lo = 0, hi = 0;
            if (row_ok) {
              if (k + 2 * d < ksz) lo = load_elem(r, k + 2 * d);
              if (k + 2 * d + 1 < ksz) hi = load_elem(r, k + 2 * d + 1);
            }
            pr[4 * q + d] = lo | (hi << 16);
          }
        }
      }
    }
  };
  auto store_stage = [&](auto slot_c, int buf) __attribute__((always_inline)) {
    uint32_t(&pr)[16] = ring[decltype(slot_c)::value];
    uint8_t* dst = my_lds0 + buf * (2 * kTile * kPitch);
    if (k_slow) {
      // pr[4q + d] = rows (2d, 2d+1) at k = kq*4 + q  ->  row i gets its four k as one 8-byte piece
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t a0 = pr[d], a1 = pr[4 + d], a2 = pr[8 + d], a3 = pr[12 + d];
        const uint2 even = make_uint2((a0 & 0xFFFFu) | (a1 << 16), (a2 & 0xFFFFu) | (a3 << 16));
        const uint2 odd = make_uint2((a0 >> 16) | (a1 & 0xFFFF0000u), (a2 >> 16) | (a3 & 0xFFFF0000u));
        *reinterpret_cast<uint2*>(dst + (rb * 8 + 2 * d) * kPitch + kq * 8) = even;
        *reinterpret_cast<uint2*>(dst + (rb * 8 + 2 * d + 1) * kPitch + kq * 8) = odd;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint4*>(dst + t7 * kPitch + q * 16) = make_uint4(pr[4 * q], pr[4 * q + 1], pr[4 * q + 2], pr[4 * q + 3]);
    }
  };

  f32x16_t acc[2][2];  // [n fragment][m fragment]
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[f][j][i] = 0.f;

  auto compute = [&](int buf) __attribute__((always_inline)) {
    const uint8_t* am = &lds[buf][0][0] + (mw * 64 + lr) * kPitch;
    const uint8_t* bn = &lds[buf][1][0] + (nw * 64 + lr) * kPitch;
#pragma unroll
    for (int t = 0; t < kKC / 16; ++t) {
      uint4 af[2], bf[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) af[j] = *reinterpret_cast<const uint4*>(am + j * 32 * kPitch + (t * 16 + h * 8) * 2);
#pragma unroll
      for (int f = 0; f < 2; ++f) bf[f] = *reinterpret_cast<const uint4*>(bn + f * 32 * kPitch + (t * 16 + h * 8) * 2);
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          // first operand = the output COLUMN side: accumulator register i of lane (lr, h) is then column
          // (i >> 2) * 8 + h * 4 + (i & 3) of row lr, four consecutive columns per register quad
          if constexpr (DT == TK_BF16)
            acc[f][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, bf[f]), __builtin_bit_cast(bf16x8_t, af[j]),
                                                                acc[f][j], 0, 0, 0);
          else
            acc[f][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, bf[f]), __builtin_bit_cast(f16x8_t, af[j]),
                                                               acc[f][j], 0, 0, 0);
        }
    }
  };

  // The slices are short (a few hundred k at most), so a tile is a handful of stages and the global-load latency is
  // what it costs: the loads run kRing stages ahead in registers, the LDS copy one stage ahead (two LDS buffers, one
  // barrier per stage).
  const int nstages = (ksz + kKC - 1) / kKC;
  if (nstages > 0) {
    static_for_ring([&](auto i_c) __attribute__((always_inline)) {
      if (decltype(i_c)::value < nstages) load_stage(i_c, decltype(i_c)::value * kKC);
    });
    store_stage(std::integral_constant<int, 0>{}, 0);
    __syncthreads();
    for (int c = 0; c < nstages; c += kRing) {
      static_for_ring([&](auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        const int cc = c + i;
        if (cc < nstages) {  // uniform
          if (cc + 1 < nstages) store_stage(std::integral_constant<int, (i + 1) % kRing>{}, (cc + 1) & 1);
          if (cc + kRing < nstages) load_stage(i_c, (cc + kRing) * kKC);  // slot i went to LDS one stage ago
          compute(cc & 1);
          __syncthreads();
        }
      });
    }
  }

  // ---- store ----
  // A lane's accumulator quad is four columns of ONE row and the 32 lanes of a fragment are 32 different rows, so
  // direct stores would touch 32 cache lines with 16 bytes each per instruction.  Instead a wave passes each 32-row
  // half of its quadrant through its own slice of LDS (the operand buffers are free now) and writes whole rows:
  // 128 bytes (16-bit outputs) or 256 bytes (fp32) of a row per 8 or 16 lanes.
  const int esize = p.y_dtype == TK_F32 ? 4 : 2;
  uint8_t* ye = p.y + (int64_t)e * p.y_stride_e * esize;
  const bool y_vec = ((p.y_stride_m * esize) % 16 == 0) && ((reinterpret_cast<uintptr_t>(ye) & 15) == 0);
  constexpr int kStagePitch = 64 * 4 + 16;  // bytes per staged row (64 columns of up to 4 bytes + pad)
  static_assert(4 * 32 * kStagePitch <= (int)sizeof(lds), "staging fits the operand buffers");
  uint8_t* stage = &lds[0][0][0] + wave * 32 * kStagePitch;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int col = f * 32 + u * 8 + h * 4;  // within the wave's 64 columns
        const float vv[4] = {acc[f][j][4 * u], acc[f][j][4 * u + 1], acc[f][j][4 * u + 2], acc[f][j][4 * u + 3]};
        if (p.y_dtype == TK_F32) {
          *reinterpret_cast<float4*>(stage + lr * kStagePitch + col * 4) = make_float4(vv[0], vv[1], vv[2], vv[3]);
        } else {
          uint32_t b[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) b[i] = p.y_dtype == TK_BF16 ? f32_to_bf16_bits(vv[i]) : f32_to_f16_bits(vv[i]);
          *reinterpret_cast<uint2*>(stage + lr * kStagePitch + col * 2) = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int lanes_per_row = 64 * esize / 16;  // 8 or 16
    const int rows_per_it = 64 / lanes_per_row;
    const int piece = lane % lanes_per_row;
    const int ncol = n0 + nw * 64 + piece * (16 / esize);
    for (int it = 0; it < 32 / rows_per_it; ++it) {
      const int r = it * rows_per_it + lane / lanes_per_row;
      const int m = m0 + mw * 64 + j * 32 + r;
      if (m >= p.M || ncol >= p.N) continue;
      const uint4 v = *reinterpret_cast<const uint4*>(stage + r * kStagePitch + piece * 16);
      uint8_t* dst = ye + ((int64_t)m * p.y_stride_m + ncol) * esize;
      if (y_vec && ncol + 16 / esize <= p.N) {
        *reinterpret_cast<uint4*>(dst) = v;
      } else {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int i = 0; i < 16 / esize && ncol + i < p.N; ++i) {
          if (esize == 4)
            reinterpret_cast<uint32_t*>(dst)[i] = w[i];
          else
            reinterpret_cast<uint16_t*>(dst)[i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// ---- both operands k-slow and aligned (the weight-gradient layout): transposition by the LDS read --------------------
// A stage is kTrK k rows x 128 m (and 128 n) in the operands' own order: the rows go from memory straight into LDS
// (buffer_load ... lds, 1 KiB = 4 k rows per wave instruction, no registers, no VALU) and ds_read_b64_tr_b16 hands a
// lane four consecutive k of ITS row, so nothing is transposed in registers.  Row pitch 256 bytes without padding (the
// DMA writes lane-contiguously): the 16-byte pieces of k row r are stored at piece ^ 4 * (r & 3), which puts the four
// rows of 64 bytes that 32 lanes of a transposing read touch on disjoint banks (^ 2 * (r & 3), disjoint for sixteen lanes only: half of the
// LDS cycles were conflicts; 16 slices of 256, 1024 x 2048 and 1024 x 1024 63 -> 57 us).  Pieces past the slice end or the matrix edge
// get an offset beyond the buffer resource; the hardware then writes zeros to LDS.
//
// What bounds it: writing y (long slices: ragged_k_long.hip).  The same kernel without its loads writes 128 x [2880, 5760] bf16 in 0.77 ms (5.5 TB/s),
// without its stores it takes 0.85 ms; together 1.13 ms (3.1 ms with the transposition in registers; 2880 x 2880: 1.5 -> 0.62).
//   * the results go through LDS so that a store instruction writes whole 128-byte lines, with the non-temporal hint
//     (pieces of 32 bytes: 1.76 ms; with the hint on such pieces 4.0, plain whole lines 1.55, whole lines with the hint 1.40) and rows of y that are no multiple
//     of a line, whose pieces begin and end inside one, by whole rows of the tile: 256 bytes an instruction have two broken lines, 128 of each wave's columns nothing
//     else (both products of a layer, us: 128 slices of 31 k, 1000 x 2000 and 1000 x 1000 365 -> 295; of 93 k, 864 x 2800 and 1400 x 864 349 -> 313; of 7 k, 1888 x 960 and
//     480 x 1888 141 -> 134; of 39 k, 2784 x 5568 and 2784 x 2784 1196 -> 1151; whole lines 140 -> 138, 2880 x 5760 and 2880 x 2880 the same);
//   * stages of 16 k, five buffers, four workgroups per CU: four fifths of the LDS are loads in flight (three buffers
//     of 32 k and three workgroups: 1.44), and a slice is padded to 16 k only;
//   * every XCD gets an eighth of EVERY slice: slices differ in length by factors, and with whole slices dealt to the
//     XCDs the longest sum decided (1.40 -> 1.21 ms); columns of tiles run first, so an XCD's eighth touches all of a and
//     an eighth of b;
//   * a tile of 128 k is two turns of the ring, and each waited for its first touch of memory behind the stream of stores: the lines are
//     asked for whole slices ahead, beyond the 128 tiles that an XCD has in flight (128 equal slices of 128 k, 258 tiles or two slices ahead,
//     1.19 -> 1.06 ms, random lengths 1.22 -> 1.13; one slice 1.17, three 1.16, every tile asking for b 1.22).
// Measured and left out (256 x 256 tiles: ragged_k_long.hip): 128 x 256 tiles, with the same ring or by persistent workgroups whose ring runs on across tiles, with loading
// and storing waves apart (1.22 to 1.40 ms); slices mixed over an XCD's workgroups (1.25).
constexpr int kTrK = 16;
constexpr int kTrBufs = 5;
constexpr int kTrOperand = kTrK * kTile * 2;   // bytes of one operand's stage
constexpr int kTrStage = 2 * kTrOperand;

// YT = element type of y (TK_BF16, TK_F16, TK_F32)
template <int DT, int YT>
__global__ __launch_bounds__(256, 4) void ragged_k_tr_kernel(const RaggedKParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kTrBufs * kTrStage];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;
  const int mw = wave & 1, nw = wave >> 1;  // the wave's 64 x 64 quadrant
  // chunks of an eighth of a slice's tiles, dealt to the XCDs in turn (workgroup b runs on XCD b % 8)
  const int per_e = p.tiles_m * p.tiles_n;
  int pid;
  {
    const int q = p.chunk, x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int round = l / q;
    pid = (round * 8 + x) * q + (l - round * q);
  }
  if (pid >= p.n_slices * per_e) return;
  const int later = pid + p.ahead;  // a tile that this XCD comes to some rounds later
  const int e = pid / per_e;
  pid -= e * per_e;
  const int tn = pid / p.tiles_m;
  const int tm = pid - tn * p.tiles_m;
  const int ksz = p.sizes[e];
  const int a_k0 = p.a_offs[e], b_k0 = p.b_offs[e];
  const int m0 = tm * kTile, n0 = tn * kTile;
  const int nst = (ksz + kTrK - 1) / kTrK;
  const uint32_t lds0 = lds_addr(lds);

  // ---- staging: a wave's instruction covers four k rows of an operand ---------------------------------------------------
  const buf_desc_t ra = make_buf_desc(p.a, p.a_bytes), rb = make_buf_desc(p.b, p.b_bytes);
  constexpr uint32_t kOutOfRange = 0x80000000u;
  const int krow = lane >> 4;                  // k row within the instruction's four
  const int piece = (lane & 15) ^ (krow * 4);  // the 16-byte piece of the row this lane fetches
  const int k_lane = wave * 4 + krow;
  static_assert(kTrK == 16, "one instruction per wave, operand and stage");
  const uint32_t a_step = (uint32_t)p.a_stride_k * 2u, b_step = (uint32_t)p.b_stride_k * 2u;
  // (a lane whose columns lie past the edge has no k in range)
  const int a_k = m0 + piece * 8 < p.M ? k_lane : ksz, b_k = n0 + piece * 8 < p.N ? k_lane : ksz;
  const uint32_t a_off = (uint32_t)(a_k0 + k_lane) * a_step + (uint32_t)(m0 + piece * 8) * 2u;
  const uint32_t b_off = (uint32_t)(b_k0 + k_lane) * b_step + (uint32_t)(n0 + piece * 8) * 2u;
  auto issue = [&](int c, uint32_t buf) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + buf + wave * 1024;
    const int k = c * kTrK;
    lds_dma16(ra, dst, a_k + k < ksz ? a_off + (uint32_t)k * a_step : kOutOfRange);
    lds_dma16(rb, dst + kTrOperand, b_k + k < ksz ? b_off + (uint32_t)k * b_step : kOutOfRange);
  };

  f32x16_t acc[2][2];  // [n fragment][m fragment]
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[f][j][i] = 0.f;

  // ---- fragment reads: lane addresses of a transposing read (row (lane & 15) >> 2 of four k, four columns) ------------
  const int l16 = lane & 15;
  const int v = ((lane >> 4) & 1) * 2 + ((l16 & 3) >> 1), swz = (l16 >> 2) * 4;
  const uint32_t rd0 = lds0 + (uint32_t)((h * 8 + (l16 >> 2)) * (kTile * 2) + (l16 & 1) * 8);
  const uint32_t frag_a[2] = {rd0 + ((mw * 8 + v) ^ swz) * 16, rd0 + ((mw * 8 + 4 + v) ^ swz) * 16};
  const uint32_t frag_b[2] = {rd0 + kTrOperand + ((nw * 8 + v) ^ swz) * 16, rd0 + kTrOperand + ((nw * 8 + 4 + v) ^ swz) * 16};
  auto compute = [&](uint32_t buf) __attribute__((always_inline)) {
    u32x4_t af[2], bf[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) af[j] = read_frag_tr(frag_a[j] + buf, kTile * 2);
#pragma unroll
    for (int f = 0; f < 2; ++f) bf[f] = read_frag_tr(frag_b[f] + buf, kTile * 2);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[f][j] = mfma_k16<DT>(bf[f], af[j], acc[f][j]);
  };

  constexpr uint32_t kLast = (kTrBufs - 1) * kTrStage;
  uint32_t rd = 0, wr = kLast;
  if (nst > 0) {
    static_for_n<kTrBufs - 1>([&](auto i_c) __attribute__((always_inline)) {
      if (decltype(i_c)::value < nst) issue(decltype(i_c)::value, decltype(i_c)::value * kTrStage);
    });
    static_assert(kTrBufs == 5, "the wait counts below list the stages that may be outstanding");
    for (int c = 0; c < nst; ++c) {
      // this wave's two pieces of stage c have landed when only those of the younger stages are outstanding
      const int ahead = nst - 1 - c;
      if (ahead >= 3)
        asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      else if (ahead == 2)
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else if (ahead == 1)
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // ... and everybody's behind the barrier; the buffer of stage c - 1 has been read
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (c + kTrBufs - 1 < nst) issue(c + kTrBufs - 1, wr);
      compute(rd);
      rd = rd == kLast ? 0 : rd + kTrStage;
      wr = wr == kLast ? 0 : wr + kTrStage;
    }
  }
  // ---- ask for lines of the later tile's operands (128 k of a's columns; of b's, which more tiles share, one tile in eight), so that L2 has them.
  // Nothing waits for these loads but the end, behind the stores.
  uint32_t ahead_a = 0, ahead_b = 0;
  if (p.ahead && later < p.n_slices * per_e) {
    const int e2 = later / per_e, in_e2 = later - e2 * per_e, tn2 = in_e2 / p.tiles_m, tm2 = in_e2 - tn2 * p.tiles_m;
    const int k = tid >> 1, col = (tid & 1) * 64;
    if (k < p.sizes[e2]) {
      const __amdgpu_buffer_rsrc_t qa = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0, p.a_bytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t qb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b), 0, p.b_bytes, 0x00020000);
      ahead_a = __builtin_amdgcn_raw_buffer_load_b32(qa, (uint32_t)(p.a_offs[e2] + k) * a_step + (uint32_t)(tm2 * kTile + col) * 2u, 0, 0);
      if ((tm2 & 7) == 0) ahead_b = __builtin_amdgcn_raw_buffer_load_b32(qb, (uint32_t)(p.b_offs[e2] + k) * b_step + (uint32_t)(tn2 * kTile + col) * 2u, 0, 0);
    }
  }
  // ---- store: a lane's accumulator quad is four columns of one row; the lane halves exchange quads, so a lane stores
  // eight consecutive columns (16-bit) or four (fp32), through a resource that drops rows past M and columns past N ----
  constexpr uint32_t ES = YT == TK_F32 ? 4 : 2;
  uint8_t* ye = p.y + (int64_t)e * p.y_stride_e * ES;
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(ye, 0, p.y_bytes, 0x00020000);
  if constexpr (YT == TK_F32) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = m0 + mw * 64 + j * 32 + lr;
      const uint32_t row = (uint32_t)m * (uint32_t)p.y_stride_m * ES;
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int n = n0 + nw * 64 + f * 32 + u * 8 + h * 4;
          const uint32_t off = (m < p.M && n < p.N) ? row + (uint32_t)n * ES : kOutOfRange;
          __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{f32_bits(acc[f][j][4 * u]), f32_bits(acc[f][j][4 * u + 1]),
                                                         f32_bits(acc[f][j][4 * u + 2]), f32_bits(acc[f][j][4 * u + 3])}, ry, off, 0, 0);
        }
    }
  } else {
    // through LDS, so that a store instruction writes four whole rows of the tile
    static_assert(kTrBufs * kTrStage >= 4 * 8192, "the four quadrants fit the operand buffers");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int j = 0; j < 2; ++j) stage_out_rows<YT>(lds + wave * 8192, j, lane, acc[0][j], acc[1][j]);
    __syncthreads();
    // a store instruction writes four rows of the whole tile: 256 bytes that lie together
    const int pc = lane & 15, n = n0 + pc * 8;
    const uint8_t* sp = lds + ((wave >> 1) + (pc >> 3) * 2) * 8192;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int r = wave * 32 + it * 4 + (lane >> 4), m = m0 + r;
      const u32x4_t q = staged_piece(sp, r & 63, pc & 7);
      const uint32_t off = (m < p.M && n < p.N) ? ((uint32_t)m * (uint32_t)p.y_stride_m + (uint32_t)n) * ES : kOutOfRange;
      __builtin_amdgcn_raw_buffer_store_b128(q, ry, off, 0, kNonTemporal);
    }
  }
  asm volatile("" ::"v"(ahead_a), "v"(ahead_b));
}

}  // namespace
}  // namespace tk

extern "C" int32_t tk_ragged_k_gemm(const tk_ragged_k_desc* d, tk_stream_t stream) {
  using namespace tk;
  if (!d) return fail(TK_ERR_INVALID, "tk_ragged_k_gemm: null descriptor");
  if (d->dtype != TK_BF16 && d->dtype != TK_F16) return fail(TK_ERR_UNSUPPORTED, "tk_ragged_k_gemm: operands must be bf16 or fp16");
  if (d->y_dtype != TK_BF16 && d->y_dtype != TK_F16 && d->y_dtype != TK_F32)
    return fail(TK_ERR_UNSUPPORTED, "tk_ragged_k_gemm: output must be bf16, fp16 or fp32");
  if (d->M < 0 || d->N < 0 || d->n_slices < 0) return fail(TK_ERR_INVALID, "tk_ragged_k_gemm: negative size");
  if (d->M == 0 || d->N == 0 || d->n_slices == 0) return TK_OK;
  if (!d->a || !d->b || !d->y || !d->slice_sizes || !d->a_slice_offs || !d->b_slice_offs)
    return fail(TK_ERR_INVALID, "tk_ragged_k_gemm: null operand");
  RaggedKParams p;
  p.a = static_cast<const uint8_t*>(d->a);
  p.a_stride_m = d->a_stride_m;
  p.a_stride_k = d->a_stride_k;
  p.b = static_cast<const uint8_t*>(d->b);
  p.b_stride_k = d->b_stride_k;
  p.b_stride_n = d->b_stride_n;
  p.y = static_cast<uint8_t*>(d->y);
  p.y_stride_e = d->y_stride_e;
  p.y_stride_m = d->y_stride_m;
  p.sizes = d->slice_sizes;
  p.a_offs = d->a_slice_offs;
  p.b_offs = d->b_slice_offs;
  p.M = d->M;
  p.N = d->N;
  p.tiles_m = (int)cdiv(d->M, kTile);
  p.tiles_n = (int)cdiv(d->N, kTile);
  p.y_dtype = d->y_dtype;
  // 16-byte loads along the contiguous dimension: base aligned and the other stride a multiple of 8 elements
  auto vec = [](const void* ptr, int64_t s_contig, int64_t s_other) {
    return s_contig == 1 && s_other % 8 == 0 && (reinterpret_cast<uintptr_t>(ptr) & 15) == 0;
  };
  p.a_vec = vec(d->a, d->a_stride_m == 1 ? d->a_stride_m : d->a_stride_k, d->a_stride_m == 1 ? d->a_stride_k : d->a_stride_m);
  p.b_vec = vec(d->b, d->b_stride_n == 1 ? d->b_stride_n : d->b_stride_k, d->b_stride_n == 1 ? d->b_stride_k : d->b_stride_n);
  int64_t grid = (int64_t)d->n_slices * p.tiles_m * p.tiles_n;
  if (grid > 0x7FFF0000) return fail(TK_ERR_UNSUPPORTED, "tk_ragged_k_gemm: grid too large");
  hipStream_t st = static_cast<hipStream_t>(stream);
  // extents (bytes from the base to one past the last element) when both operands are k-slow and within 2 GiB
  const bool k_slow_both = d->a_stride_m == 1 && d->b_stride_n == 1 && d->a_stride_k > 0 && d->b_stride_k > 0;
  const int64_t a_extent = d->a_k_extent * d->a_stride_k * 2, b_extent = d->b_k_extent * d->b_stride_k * 2;
  const bool fast = k_slow_both && p.a_vec && p.b_vec && d->M % 8 == 0 && d->N % 8 == 0 && d->a_k_extent > 0 && d->b_k_extent > 0 &&
                    a_extent < (int64_t(1) << 31) && b_extent < (int64_t(1) << 31) && d->M <= d->a_stride_k && d->N <= d->b_stride_k;
  const int64_t es = d->y_dtype == TK_F32 ? 4 : 2, y_extent = ((int64_t)(d->M - 1) * d->y_stride_m + d->N) * es;
  const bool y_ok = d->y_stride_m >= d->N && y_extent < (int64_t(1) << 31) && d->y_stride_m * es % 16 == 0 && d->y_stride_e * es % 16 == 0 &&
                    (reinterpret_cast<uintptr_t>(d->y) & 15) == 0;
  p.a_bytes = fast ? (uint32_t)a_extent : 0;
  p.b_bytes = fast ? (uint32_t)b_extent : 0;
  p.y_bytes = y_ok ? (uint32_t)y_extent : 0;
  auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), 0, st, p); };
  const bool bf16 = d->dtype == TK_BF16;
  if (fast && y_ok) {
    const int per_e = p.tiles_m * p.tiles_n;
    p.n_slices = d->n_slices;
    // (rows past M of a long slice's last tiles go by offsets beyond the resource, which may not wrap)
    const bool long_runs = (int64_t)(d->M + 256) * d->y_stride_m * es < (int64_t(1) << 32);
    const int tile = long_runs ? ragged_k_tile(std::min(d->a_k_extent, d->b_k_extent) / d->n_slices, d->M, d->N, d->n_slices) : 0;
    if (tile) return ragged_k_launch_long(p, d->dtype, tile, st);
    p.chunk = per_e >= 8 ? per_e / 8 : 1;
    // An XCD's part of a slice below 32 tiles: lines asked for six and more slices ahead are gone again or not yet of use (both products of a layer, all by this kernel,
    // 16384 rows, 128 slices, 15 and 8 tiles: 165 us without against 173; 23 and 12: 385 / 391; 36 and 18: 545 / 556; 31 and 16: 420 / 420;
    // 33 and 17: 478 / 477; 45 and 23: 685 / 659; 68 and 35: 1010 / 970).  Fewer than 64 slices: what there is to wait for is less (2880 x 5760 and
    // 2880 x 2880, 32 slices of 128 389 / 393, 8 of 2048 933 / 942; 2048 x 4096 and 2048 x 2048, 64 slices of 128 472 / 462).
    p.ahead = p.chunk >= 32 && d->n_slices >= 64 ? 8 * p.chunk * (int)cdiv(192, p.chunk) : 0;
    const int64_t chunks = cdiv((int64_t)d->n_slices * per_e, p.chunk);
    grid = cdiv(chunks, 8) * 8 * p.chunk;
    auto with_y = [&](auto dt) {
      constexpr int DT = decltype(dt)::value;
      if (d->y_dtype == TK_BF16)
        launch(ragged_k_tr_kernel<DT, TK_BF16>);
      else if (d->y_dtype == TK_F16)
        launch(ragged_k_tr_kernel<DT, TK_F16>);
      else
        launch(ragged_k_tr_kernel<DT, TK_F32>);
    };
    bf16 ? with_y(std::integral_constant<int, TK_BF16>{}) : with_y(std::integral_constant<int, TK_F16>{});
    return check_launch("ragged_k_tr_kernel");
  }
  bf16 ? launch(ragged_k_gemm_kernel<TK_BF16>) : launch(ragged_k_gemm_kernel<TK_F16>);
  return check_launch("ragged_k_gemm_kernel");
}
