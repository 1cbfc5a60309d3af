// A whole decode-sized MoE FFN layer in ONE launch: router -> gather-GEMM (+bias, swiglu) -> scatter-GEMM (+bias,
// gate weight) -> top-k combine, for a handful of tokens (T * k <= 256 routed rows) over tiled MXFP4 expert weights.
//
// At these sizes the layer is a stream of the active experts' weights (13 MB per expert at the gpt-oss shape) read
// once from HBM; three launches spend a third of their time on launch boundaries and on the serial router in front
// of the first weight byte.  Here the grid is persistent and co-resident (one workgroup per CU):
//
//   1. EVERY workgroup routes all T tokens itself (the logits are a few KiB): top-k by wave-wide max rounds, softmax,
//      expert histogram, stable expert-sorted row order - into LDS, no global round trip, no dependence on others.
//   2. The work is cut into units = (active expert, 16-row block, one or two 32-column weight fragments) of GEMM 1 followed by
//      those of GEMM 2; every workgroup takes an equal contiguous share of each list, derived from the LDS tables.
//   3. The NW waves of a workgroup share the K-stages of a unit (XS = 1 to 3 each; three: consecutive ones, so that the sums are those of
//      K / 384 slices added in order; one or two: in turn, which leaves no wave idle); a wave keeps its part of the
//      block's activation rows in REGISTERS for as long as the (expert, row block) stays the same, so the inner loop
//      is: 2 KiB weight block global -> registers (ring of three or four units), e2m1 -> bf16 in registers, 16x16x32 MFMA.
//      The waves' sums meet in LDS once per unit (one barrier); four of the waves, the even ones of an even unit and the odd ones of an odd one, add them and run the
//      epilogue.  (One wave in turn: its next unit started late, and the others met it at the barrier; all waves: a quarter of a microsecond of each
//      one's time.  49 tokens, 64 experts, top 2, d 1952, d_ff 960: 60.7 / 59.4 with four / 59.9 us; 60 tokens, 96 experts, top 4, 2048: 69.5 / 68.9 / 70.1;
//      61 tokens, 128 experts, top 4, 2880, with favourites: 116.1 / 114.5 / 116.0.)
//   4. GEMM 1 writes its swiglu'd rows (bf16) to a scratch tensor h with write-through stores; a workgroup that has
//      finished its GEMM-1 share counts its units in at a counter per row block.  GEMM-2 units of a block wait for that
//      counter (their weight blocks are already on their way) and read h around the L2 (the eight XCDs' L2s are not
//      coherent with each other).
//   5. GEMM 2 writes gate-weighted rows to y [T*k, N]; when a workgroup has finished its share it counts every
//      (token, fragment) it wrote in, and whoever completes a token's k rows sums them in j order in fp32 (what
//      `reduce` does after the reference's scatter, reduce.py:1143-1165) and writes the token's output row.
//   6. The last workgroup to finish clears the counters, so the workspace is ready for the next launch.
//
// Every wait is bounded: a spin that exceeds `spin_limit` polls raises the error word of the workspace and goes on
// (the result is then wrong, but every wave exits).
#include "decode_params.h"
#include "gemm_common.h"
#include "route_common.h"

namespace tk {
namespace {

constexpr int kDecMaxRows = TK_DECODE_MAX_ROWS;        // T * k
constexpr int kDecMaxExperts = TK_DECODE_MAX_EXPERTS;  // one expert per thread in the placement pass
constexpr int kDecMaxUnits = 192;                      // units (of one fragment) of a workgroup (the host bounds it)
constexpr int kDecNW = 8;                              // waves per workgroup, which share a unit's K-stages
constexpr int kDecXS = 3;                              // K-stages (of 128) of a wave at most: K <= NW * XS * 128 = 3072
constexpr int kDecBlockStride = 32;                    // words between two row blocks' counters (a cache line each)
constexpr int kDecBlockWords = (kDecMaxRows + kDecMaxRows / 16) * kDecBlockStride;  // 16-row blocks: at most min(E, R) + R / 16

struct DecUnit {
  const uint8_t* w;  // first K-stage of the unit's weight fragment
  const uint8_t* s;
  int32_t key;       // phase << 24 | expert slot a << 8 | row block
  int32_t frag;      // first column fragment F
  int32_t once;      // its expert has one row block only
};

// XS: K-stages of a wave, FPU: column fragments of a unit.  A unit costs its chain (weights, products, sums through LDS, barrier) whatever its
// bytes, so short K take fewer stages a wave, which leaves registers for a deeper ring or for two fragments a unit.
template <int XS_, int FPU_>
struct DecCfg {
  static constexpr int XS = XS_, FPU = FPU_;
  static constexpr int STAGE0 = XS == 3 ? 3 : 1, STEP = XS == 3 ? 1 : kDecNW;  // wave w's stages: w * STAGE0 + j * STEP
  static constexpr int RING = XS * FPU >= 3 ? 3 : 4;      // units of weight blocks a wave holds or has requested
  static constexpr int UNITS = kDecMaxUnits / FPU;        // of one workgroup
  static constexpr int COLS = 32 * FPU;
};

#ifdef TK_DEC_STAMPS
__device__ long long dec_stamps[1024][20];
#define DEC_STAMP(n) do { if (threadIdx.x == 0) dec_stamps[blockIdx.x][n] = (long long)__builtin_amdgcn_s_memrealtime(); } while (0)
// end of unit i's K loop in every workgroup (rows 512 + 2 * workgroup of the table, 20 columns x 2 rows each)
#define DEC_UNIT_STAMP(i) do { if (threadIdx.x == 0 && blockIdx.x < 256 && (i) < 40) dec_stamps[512 + blockIdx.x * 2 + (i) / 20][(i) % 20] = (long long)__builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define DEC_UNIT_STAMP(i) do {} while (0)
#define DEC_STAMP(n) do {} while (0)
#endif

// x of another lane of the lane's four (DPP quad permutation)
template <int PERM>
__device__ __forceinline__ float quad_swap(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), PERM, 0xF, 0xF, true));
}

constexpr int kNonTemporalLoad = 2;

constexpr int kThrough = 1 | 16;  // aux bits of the buffer instructions: sc0 | sc1 (write through / read around the L2)

template <int VPL, int XS_, int FPU_, int FETCH>
__global__ __launch_bounds__(kDecNW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_decode_layer_kernel(const DecodeParams p) {
  typedef DecCfg<XS_, FPU_> C;
  constexpr int NW = kDecNW, XS = C::XS, FPU = C::FPU, NT = NW * 64;
  typedef Frag<16> FR;
  __shared__ int16_t eid_s[kDecMaxRows];      // expert of flat entry f = t*k + j
  __shared__ float gate_s[kDecMaxRows];       // its gate value
  __shared__ int16_t rowflat_s[kDecMaxRows];  // flat entry of expert-sorted row
  __shared__ int32_t hist_s[kDecMaxExperts];
  __shared__ int32_t offs_s[kDecMaxExperts + 1];  // first expert-sorted row of expert e
  __shared__ int16_t act_s[kDecMaxExperts];       // a -> expert id, active experts in ascending order
  __shared__ int32_t bpre_s[kDecMaxExperts + 1];  // a -> 16-row blocks of the active experts before a
  __shared__ int32_t misc_s[4];                   // [0] number of active experts
  __shared__ DecUnit tab_s[C::UNITS + C::RING];
  // partial sums of a unit: [unit parity][wave][row][column], the 16-byte pieces of row r stored at piece ^ (r & 7): neither the waves' quads nor the
  // rows of columns that a wave sums conflict in a bank
  __shared__ __attribute__((aligned(16))) float red_s[2][NW][16][C::COLS];
  __shared__ __attribute__((aligned(16))) float bias_s[C::UNITS][C::COLS];  // bias of a unit's columns
  __shared__ u32x4_t xst_s[NW][4][64];  // per wave: one K-stage of a row block's activations on its way into MFMA order

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, kg = lane >> 4;
  const int T = p.T, E = p.E, k = p.k, R = T * k;
  const int G = (int)gridDim.x;

  DEC_STAMP(0);
  // ---- 1. routing, by every workgroup for itself ----------------------------------------------------------
  // Sixteen lanes (one DPP row) own a token, four tokens per wave at a time; lane l of the row holds the VPL
  // consecutive experts l*VPL .. l*VPL+VPL-1 as order-preserving keys.  A round = the row's largest key still in the
  // running (in-lane maximum, then four DPP steps inside the row) and the LOWEST expert index holding it (same again
  // with a minimum): ties go to the lower expert, as the reference's packed sort key does
  // (topk_details/_topk_forward.py:27-35,61).  No lane leaves its row, so the four tokens cost what one costs.
  // [token word][expert]: bit t of word w = token 32 w + t chose the expert.  (Experts along the rows: in the other order the
  // lanes of the counting pass below, which own neighbouring experts, all met in one LDS bank.)
  int32_t(*mask_s)[kDecMaxExperts] = reinterpret_cast<int32_t(*)[kDecMaxExperts]>(&red_s[0][0][0][0]);
  {
    const int l16 = lane & 15, sub = lane >> 4;
    for (int row0 = 0; row0 < T; row0 += NW * 4) {
      const bool wave_has_rows = row0 + wave * 4 < T;  // (uniform) a wave without tokens stays out of the others' way
      if (!wave_has_rows && row0 > 0) break;
      const int row = row0 + wave * 4 + sub;
      const bool row_ok = row < T;
      uint32_t key[VPL];
      uint32_t ret = 0;  // bit i: key[i] is out of the running
#pragma unroll
      for (int i = 0; i < VPL; ++i) {
        const int e = l16 * VPL + i;
        float f = 0.f;
        if (row_ok && e < E) {
          const int64_t at = (int64_t)row * p.logits_stride + e;
          f = p.logits_is_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(p.logits)[at]) : static_cast<const float*>(p.logits)[at];
        }
        key[i] = ordered_key(f);
        ret |= (e >= E ? 1u : 0u) << i;
      }
      if (row0 == 0) {  // the masks are cleared while the first logits are on their way (every wave comes through here)
        for (int i = tid; i < kDecMaxExperts * ((T + 31) >> 5); i += NT) (&mask_s[0][0])[i] = 0;
        __syncthreads();
        DEC_STAMP(17);
      }
      if (!wave_has_rows) break;
      if (row0 == 0 && key[0] == 0x12345u) DEC_STAMP(9);  // (never true: makes the stamp below wait for the logits)
      if (row0 == 0) DEC_STAMP(18);
      uint32_t sel_key[2] = {0u, 0u};
      int sel_idx[2] = {0, 0};
      uint32_t key0 = 0;
      row16_topk<VPL>(key, ret, k, l16, sel_key, sel_idx, key0);
      if (row0 == 0) DEC_STAMP(19);
      // softmax over the k kept logits (fp32): z = exp(v - max) / sum
      float outv[2], z[2];
      const float vmax = key_to_float(key0);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool have = l16 + 16 * q < k;
        outv[q] = key_to_float(sel_key[q]);
        z[q] = have ? expf(outv[q] - vmax) : 0.f;
      }
      if (p.apply_softmax) {
        const float sum = row16_sum_f32(z[0] + z[1]);
        outv[0] = z[0] / sum;
        outv[1] = z[1] / sum;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int j = l16 + 16 * q;
        if (row_ok && j < k) {
          int e = sel_idx[q];
          e = e < 0 ? 0 : (e < E ? e : E - 1);  // (k <= E: every round finds a column)
          eid_s[row * k + j] = (int16_t)e;
          gate_s[row * k + j] = outv[q];
          atomicOr(&mask_s[row >> 5][e], 1 << (row & 31));
          if (blockIdx.x == 0) {
            if (p.indx_out) p.indx_out[row * k + j] = (int16_t)e;
            if (p.vals_out) p.vals_out[row * k + j] = outv[q];
          }
        }
      }
    }
  }
  __syncthreads();
  DEC_STAMP(1);
  // ---- rows per expert, expert offsets, the list of active experts and their row blocks (wave 0) ----------
  const int tw = (T + 31) >> 5;  // token words in use
  if (wave == 0) {
    constexpr int PER = VPL * 16 / 64;  // experts per lane (the kernel's variant covers VPL * 16 experts)
    int cnt[PER];
    int rows = 0, blks = 0, acts = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane * PER + i;
      int c = 0;
      if (e < E)
        for (int w = 0; w < tw; ++w) c += __builtin_popcount((uint32_t)mask_s[w][e]);
      cnt[i] = c;
      rows += c;
      blks += (c + 15) >> 4;
      acts += c > 0 ? 1 : 0;
    }
    const int prow = wave_scan_i32(rows), pblk = wave_scan_i32(blks), pact = wave_scan_i32(acts);  // inclusive, over the lanes
    int r0 = prow - rows, b0 = pblk - blks, a0 = pact - acts;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane * PER + i;
      if (e < E) {
        hist_s[e] = cnt[i];
        offs_s[e] = r0;
        if (cnt[i] > 0) {
          act_s[a0] = (int16_t)e;
          bpre_s[a0] = b0;
          ++a0;
        }
        r0 += cnt[i];
        b0 += (cnt[i] + 15) >> 4;
      }
    }
    if (lane == 63) {
      offs_s[E] = prow;
      bpre_s[pact] = pblk;
      misc_s[0] = pact;
    }
  }
  __syncthreads();
  // ---- expert-sorted row order (stable): entry (t, j) of expert e goes behind the entries of e from earlier tokens ----
  for (int f = tid; f < R; f += NT) {
    const int e = eid_s[f], t = f / k;
    int rank = 0;
    for (int w = 0; w < (t >> 5); ++w) rank += __builtin_popcount((uint32_t)mask_s[w][e]);
    rank += __builtin_popcount((uint32_t)mask_s[t >> 5][e] & ((1u << (t & 31)) - 1u));
    rowflat_s[offs_s[e] + rank] = (int16_t)f;
  }
  const int A = misc_s[0];
  const int nblk = bpre_s[A];
  // ---- 2. this workgroup's share of the unit lists ---------------------------------------------------------
  // unit uu of a list = (row block uu / nfr, fragment uu % nfr): a workgroup's run stays on one row block, whose
  // activation rows its waves keep in registers.  The row blocks are cut into two halves and every workgroup works
  // through four runs: GEMM 1 of the first half, GEMM 1 of the second, GEMM 2 of the first, GEMM 2 of the second.
  // When a workgroup reaches a GEMM-2 run, the rows of h it needs were finished (by all workgroups) a whole run
  // earlier, so the hand-over between the GEMMs costs no waiting.
  const int bh = (nblk + 1) >> 1;  // row blocks of the first half
  // (32-bit arithmetic: nblk <= 272 and nfr1 + nfr2 <= 288, so G * (U1 + U2) stays below 2^25; a 64-bit division is
  // a hundred instructions, and a dozen of them stood between the routing and the first weight request)
  const int nu1 = (p.nfr1 + FPU - 1) / FPU, nu2 = (p.nfr2 + FPU - 1) / FPU;  // units of a row block
  const int U1 = nblk * nu1, U2 = nblk * nu2;
  const int L0 = bh * nu1, L1 = U1 - L0, L2 = bh * nu2, L3 = U2 - L2;
  const int wg = blockIdx.x;
  auto udiv = [](int a, int b) -> int { return (int)((uint32_t)a / (uint32_t)b); };
  // Shares.  The four runs are cut as one list: cut i of a run = floor(i * (S + L) / G) - floor(i * S / G), S = the
  // units of the runs in front of it, L its own, so that what a workgroup has got from the runs so far is
  // floor((i + 1) * S / G) - floor(i * S / G) whatever the remainders were: a workgroup's units of the whole layer
  // differ by at most one from any other's, and so do its units of GEMM 1 (the GEMM-2 runs wait for everybody's
  // GEMM-1 runs).  A unit of either GEMM costs the same, and with a dozen units per workgroup one more in every run is a
  // quarter more work.  The cuts grow with i when L >= 2 G (their increment is at least L / G - 2); a shorter run is cut
  // evenly by itself and the list starts again with it.
  int S = 0;
  auto share = [&](int L, int& cut_b, int& cut_e) {
    if (S != 0 && L < 2 * G) S = 0;
    cut_b = udiv(wg * (S + L), G) - udiv(wg * S, G);
    cut_e = udiv((wg + 1) * (S + L), G) - udiv((wg + 1) * S, G);
    S += L;
  };
  int c0b, c1b, c0e, c1e, c2b, c3b, c2e, c3e;
  share(L0, c0b, c0e);
  share(L1, c1b, c1e);
  share(L2, c2b, c2e);
  share(L3, c3b, c3e);
  const int r0b = c0b, r0e = c0e, r1b = L0 + c1b, r1e = L0 + c1e;
  const int r2b = c2b, r2e = c2e, r3b = L2 + c3b, r3e = L2 + c3e;
  int nr0 = r0e - r0b, nr1 = r1e - r1b, nr2 = r2e - r2b, nr3 = r3e - r3b;
  if (nr0 + nr1 + nr2 + nr3 > C::UNITS) {  // (the host's bound rules this out)
    if (tid == 0) atomicOr(&p.sync[1], 2);
    nr0 = nr0 < C::UNITS ? nr0 : C::UNITS;
    nr1 = nr1 < C::UNITS - nr0 ? nr1 : C::UNITS - nr0;
    nr2 = nr2 < C::UNITS - nr0 - nr1 ? nr2 : C::UNITS - nr0 - nr1;
    nr3 = nr3 < C::UNITS - nr0 - nr1 - nr2 ? nr3 : C::UNITS - nr0 - nr1 - nr2;
  }
  const int n1 = nr0 + nr1, n2 = nr2 + nr3;
  const int n_units = n1 + n2;
  // (no barrier here: the table below is built from the scan's results, like the row order above)
  for (int i = tid; i < n_units + C::RING; i += NT) {
    DecUnit u;
    if (i >= n_units) {  // behind the last unit nothing is fetched
      u.w = p.w1;
      u.s = p.w1s;
      u.key = -1;
      u.frag = 0;
      u.once = 1;
    } else {
      const bool ph2 = i >= n1;
      const int uu = i < nr0 ? r0b + i : i < n1 ? r1b + (i - nr0) : i < n1 + nr2 ? r2b + (i - n1) : r3b + (i - n1 - nr2);
      const int nu = ph2 ? nu2 : nu1;
      const int nst = ph2 ? p.nst2 : p.nst1;
      const int B = udiv(uu, nu), F = (uu - B * nu) * FPU;
      int lo = 0, hi = A;  // last a with bpre[a] <= B
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (bpre_s[mid] <= B) lo = mid; else hi = mid;
      }
      const int a = lo, rb = B - bpre_s[a];
      const int e = act_s[a];
      u.w = (ph2 ? p.w2 + (int64_t)e * p.w2_stride_e : p.w1 + (int64_t)e * p.w1_stride_e) + (int64_t)F * nst * 2048;
      u.s = (ph2 ? p.w2s + (int64_t)e * p.w2s_stride_e : p.w1s + (int64_t)e * p.w1s_stride_e) + (int64_t)F * nst * 128;
      u.key = ((ph2 ? 2 : 1) << 24) | (a << 8) | rb;
      u.frag = F;
      u.once = bpre_s[a + 1] - bpre_s[a] == 1;
    }
    tab_s[i] = u;
  }
  __syncthreads();  // (the token masks are dead from here on: their memory becomes the reduction buffers)
  DEC_STAMP(2);

  // ---- 3. the stream ----------------------------------------------------------------------------------------
  // lane (lr, kg): weight columns g*16 + lr of the fragment, k-block kg (32 k = 16 packed bytes) of every stage;
  // this wave's stages of a unit are wave * STAGE0 + j * STEP
  const uint32_t wlane = (uint32_t)((kg & 1) * 1024 + ((kg >> 1) * 32 + lr) * 16);
  const uint32_t slane = (uint32_t)(lr * 4);
  // weight registers: RD sets of XS stages; unit i lives in set i % RD and, stage by stage as it is consumed, is
  // replaced by unit i + RD.  A wave's requests are answered in order, one unit per unit time, so a block must be
  // requested RD unit times before it is used: with a loaded memory latency of about 4 us and three stages a wave, two sets bound a unit at
  // 2 us (what was measured), three at 1.3 us, which is below what HBM delivers (19 KiB per wave on its way).  The shorter units of less K have 17 KiB on
  // their way (four sets of one stage and two fragments, or of two and one) or 25.5 (three of two and two).
  constexpr int RD = C::RING;
  const __amdgpu_buffer_rsrc_t hrsrc = __builtin_amdgcn_make_buffer_rsrc(p.h, 0, (uint32_t)((int64_t)R * p.K2 * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(p.y, 0, (uint32_t)((int64_t)R * p.N2 * 2), 0x00020000);
  const float nalpha_log2e = -p.alpha * 1.4426950408889634f;
  const float limit = p.has_limit ? p.limit : INFINITY;

  // table entries are the same for every lane: keep them in scalar registers
  auto uniform_unit = [&](int i) __attribute__((always_inline)) -> DecUnit {
    const DecUnit v = tab_s[i];
    const uint64_t w = (uint64_t)v.w, sc = (uint64_t)v.s;
    DecUnit u;
    u.w = (const uint8_t*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(w >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)w));
    u.s = (const uint8_t*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(sc >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)sc));
    u.key = __builtin_amdgcn_readfirstlane(v.key);
    u.frag = __builtin_amdgcn_readfirstlane(v.frag);
    u.once = XS == 3 ? __builtin_amdgcn_readfirstlane(v.once) : 0;
    return u;
  };
  // counts GEMM-1 units [from, to) of this workgroup in at their row blocks' counters (unit u belongs to block u / nu1)
  auto signal_blocks = [&](int ub, int ue) __attribute__((always_inline)) {
    if (ue > ub) {
      const int b_first = udiv(ub, nu1), b_last = udiv(ue - 1, nu1);
      for (int b = b_first + tid; b <= b_last; b += NT) {
        const int lo = b * nu1, hi = lo + nu1;
        const int from = lo > ub ? lo : ub, to = hi < ue ? hi : ue;
        __hip_atomic_fetch_add(&p.sync[2 + b * kDecBlockStride], to - from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  };
  // ---- the biases of this workgroup's units, to LDS: requested in front of the first weight blocks (what is requested behind them is answered behind
  // them, and the wait would be one for the whole ring), written when the first activations have come.  Four values a thread cover 2048 columns; more take
  // another round.  As two halves (of a bf16 bias the same one twice), from the activations where there is nothing: a load under a condition is waited for at its end. ----
  constexpr int BPT = 4, kBiasRound = BPT * NT / C::COLS;  // values of a thread, units of a round
  uint64_t b1 = (uint64_t)p.b1, b2 = (uint64_t)p.b2;
  int64_t b1_stride = p.b1_stride_e, b2_stride = p.b2_stride_e;
  int b1_f32 = p.b1_is_f32, b2_f32 = p.b2_is_f32, n_of1 = p.N1, n_of2 = p.N2;
  // (opaque: a choice between two of the kernel's arguments by a lane's GEMM becomes a load of them otherwise)
  asm volatile("" : "+s"(b1), "+s"(b2), "+s"(b1_stride), "+s"(b2_stride), "+s"(b1_f32), "+s"(b2_f32), "+s"(n_of1), "+s"(n_of2));
  uint16_t bias_lo[BPT], bias_hi[BPT];
  auto bias_fetch = [&](int first_unit) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const int idx = first_unit * C::COLS + q * NT + tid, ui = idx / C::COLS;
      const DecUnit u = tab_s[ui < n_units ? ui : 0];
      const bool ph2 = (u.key >> 24) == 2, f32 = ph2 ? b2_f32 : b1_f32;
      const int n = u.frag * 32 + idx % C::COLS;
      const uint64_t bp = ph2 ? b2 : b1;
      const bool have = bp && n < (ph2 ? n_of2 : n_of1);
      const int64_t el = (int64_t)act_s[(u.key >> 8) & 0xFFFF] * (ph2 ? b2_stride : b1_stride) + n;
      const uint64_t at = have ? bp + ((uint64_t)el << (f32 ? 2 : 1)) : (uint64_t)p.x;
      bias_lo[q] = *(const __attribute__((address_space(1))) uint16_t*)at;
      bias_hi[q] = *(const __attribute__((address_space(1))) uint16_t*)(have && f32 ? at + 2 : at);
    }
  };
  auto bias_park = [&](int first_unit) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      const int idx = first_unit * C::COLS + q * NT + tid, ui = idx / C::COLS;
      if (ui < n_units) {
        const DecUnit u = tab_s[ui];
        const bool ph2 = (u.key >> 24) == 2, f32 = ph2 ? b2_f32 : b1_f32;
        const bool have = (ph2 ? b2 : b1) && u.frag * 32 + idx % C::COLS < (ph2 ? n_of2 : n_of1);
        const uint32_t hi = bias_hi[q];
        (&bias_s[0][0])[idx] = bits_f32(!have ? 0u : f32 ? hi << 16 | bias_lo[q] : hi << 16);
      }
    }
  };
  for (int u0 = kBiasRound; u0 < n_units; u0 += kBiasRound) {
    bias_fetch(u0);
    bias_park(u0);
  }
  bool signalled0 = nr0 == 0, signalled = n1 == 0;  // see below
  auto stream = [&](auto mode_c) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value;
    u32x4_t wr[RD][XS][FPU][2];
    uint32_t sr[RD][XS][FPU][2];
    u32x4_t xr[XS][4];
    // (Stages and fragments past the unit's last are past the resource's end: zeros, and no memory is asked for them.  No branch around a load: the compiler's wait
    // counts stay exact only in straight-line code.)
    uint32_t w_at[XS], s_at[XS];
#pragma unroll
    for (int j = 0; j < XS; ++j) w_at[j] = wlane + (uint32_t)(wave * C::STAGE0 + j * C::STEP) * 2048u, s_at[j] = slane + (uint32_t)(wave * C::STAGE0 + j * C::STEP) * 128u;
    auto load_w = [&](auto h_c, int j, const DecUnit& u, int nst, int nfr) __attribute__((always_inline)) {
      constexpr int H = decltype(h_c)::value;
      auto fetch = [&](auto aux_c) __attribute__((always_inline)) {
        constexpr int AUX = decltype(aux_c)::value;
#pragma unroll
        for (int f = 0; f < FPU; ++f) {
          const int stages = FPU == 1 || u.frag + f < nfr ? nst : 0;
          const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(u.w + (int64_t)f * nst * 2048), 0, stages * 2048, 0x00020000);
          const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(u.s + (int64_t)f * nst * 128), 0, stages * 128, 0x00020000);
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            wr[H][j][f][g] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, w_at[j] + g * 256, 0, AUX);
            sr[H][j][f][g] = __builtin_amdgcn_raw_buffer_load_b32(srsrc, s_at[j] + g * 64, 0, AUX);
          }
        }
      };
      if (MODE == kFetchOnce || (MODE == kFetchEither && u.once))
        fetch(template_int<kNonTemporalLoad>{});
      else
        fetch(template_int<0>{});
    };
    auto unit_nst = [&](const DecUnit& u) __attribute__((always_inline)) -> int { return u.key < 0 ? 0 : (u.key >> 24) == 2 ? p.nst2 : p.nst1; };
    auto unit_nfr = [&](const DecUnit& u) __attribute__((always_inline)) -> int { return (u.key >> 24) == 2 ? p.nfr2 : p.nfr1; };
    // This wave's stages of a row block's activation rows: x through the expert-sorted order for GEMM 1, h for GEMM 2.
    // The MFMA wants row lr's k-block kg in lane (lr, kg): loaded that way, the sixteen lanes that one pass of a load
    // serves touch sixteen rows, i.e. sixteen cache lines for 16 bytes each.  So the rows are loaded four lanes to a row
    // (lane = row * 4 + chunk: 64 contiguous bytes per row and instruction, rows past the block's last dropped, not
    // repeated) and turned into MFMA order through a 4 KiB buffer of the wave's own in LDS, one K-stage at a time
    // (LDS operations of a wave execute in order; 16-byte chunks swizzled by the row so that neither side conflicts).
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.x), 0, p.x_bytes, 0x00020000);
    auto x_request = [&](auto ph_c, const DecUnit& u) __attribute__((always_inline)) {
      constexpr int ph = decltype(ph_c)::value;  // 1: rows of x, 2: rows of h
      const int a = (u.key >> 8) & 0xFFFF, rb = u.key & 0xFF;
      const int e = act_s[a];
      const int cnt = hist_s[e];
      const int row0 = offs_s[e] + rb * 16;
      const int rows = cnt - rb * 16 < 16 ? cnt - rb * 16 : 16;
      const int r = lane >> 2, c = lane & 3;
      const bool valid = r < rows;
      const int K = ph == 2 ? p.K2 : p.K1;
      // first k of this lane in its wave's slice (opaque: otherwise the twelve addresses below are computed once, ahead
      // of the loop, and parked in scratch memory, which turns every reload into a chain of dependent memory round trips)
      int kb = wave * (C::STAGE0 * 128) + c * 8;
      asm volatile("" : "+v"(kb));
      uint32_t base;
      if constexpr (ph == 2) {
        base = (uint32_t)(row0 + r) * (uint32_t)(p.K2 * 2);
      } else {
        const int token = rowflat_s[row0 + (valid ? r : 0)] / k;
        base = (uint32_t)token * (uint32_t)(p.x_stride * 2);
      }
#pragma unroll
      for (int j = 0; j < XS; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int k0 = kb + j * (C::STEP * 128) + q * 32;
          // past K the weights are zero (padding, stages past the last): zeros will do
          const uint32_t off = (valid && k0 < K) ? base + (uint32_t)k0 * 2u : kDroppedStore;
          if constexpr (ph == 2)
            xr[j][q] = __builtin_amdgcn_raw_buffer_load_b128(hrsrc, off, 0, kThrough);
          else
            xr[j][q] = __builtin_amdgcn_raw_buffer_load_b128(xrsrc, off, 0, 0);
        }
    };
    auto x_settle = [&]() __attribute__((always_inline)) {
      const int r = lane >> 2, c = lane & 3;
      const int wpos = r * 4 + (c ^ ((r >> 2) & 3));
#pragma unroll
      for (int j = 0; j < XS; ++j) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q) xst_s[wave][q][wpos] = xr[j][q];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < 4; ++t) xr[j][t] = xst_s[wave][kg][lr * 4 + (t ^ ((lr >> 2) & 3))];
      }
    };
    int cur_key = 0;
    if (n_units > 0) {
      bias_fetch(0);
      // the first unit's activation slice is requested in front of the weight blocks (a wave's requests are answered in
      // order, and the units of weight blocks primed below keep the memory system busy for microseconds)
      const DecUnit first = uniform_unit(0);
      const bool x_first = (first.key >> 24) == 1;
      if (x_first) {
        x_request(std::integral_constant<int, 1>{}, first);
        cur_key = first.key;
      }
      static_for<0, RD>([&](auto h_c) __attribute__((always_inline)) {
        const DecUnit u = uniform_unit(decltype(h_c)::value);
#pragma unroll
        for (int j = 0; j < XS; ++j) load_w(h_c, j, u, unit_nst(u), unit_nfr(u));
      });
      // (here, in straight-line code behind the requests, the wait in front of the LDS writes counts the weight blocks
      // out: behind the bias loops below it would be a wait for everything requested so far)
      if (x_first) x_settle();
      bias_park(0);
    }
    // A finished GEMM-1 run is counted in without draining the wave's memory queue.  A wave's loads and stores complete
    // in issue order.  The epilogue of a run's last unit stores its rows of h right behind that unit's barrier; the
    // next unit opens another row block (or the other GEMM), so EVERY wave starts it by fetching new activation rows
    // and consumes them in its K loop.  Behind that unit's barrier all stores of the finished run have therefore
    // reached memory, and the run is counted in there.  (A wait that comes earlier than that, possible only for a
    // workgroup with next to no units, drains the queue and counts in first: a workgroup must never wait for rows
    // that it has not counted in itself.)
    auto unit_body = [&](auto h_c, int i) __attribute__((always_inline)) {
      constexpr int H = decltype(h_c)::value;
      const DecUnit cur = uniform_unit(i);
      const DecUnit nxt = uniform_unit(i + RD);  // the unit that takes over this set of weight registers
      const int ph = cur.key >> 24, a = (cur.key >> 8) & 0xFFFF, rb = cur.key & 0xFF;
      const int e = act_s[a];
      const int cnt = hist_s[e];
      const int row0 = offs_s[e] + rb * 16;                       // first expert-sorted row of the block
      const int rows = cnt - rb * 16 < 16 ? cnt - rb * 16 : 16;  // valid rows of the block
      if (i == 1) DEC_STAMP(3);
      if (i == n1) DEC_STAMP(4);
      if (cur.key != cur_key) {
        cur_key = cur.key;
        // ---- a new (expert, row block): this wave's stages of its activation rows go into registers ----
        if (ph == 2) {
          const int blk = bpre_s[a] + rb;  // a block of the first half was computed by run 0 alone
          if (!signalled0 || (blk >= bh && !signalled)) {  // (uniform) see above: count in what this workgroup itself still owes
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (!signalled0) signal_blocks(r0b, r0b + nr0);
            if (!signalled) signal_blocks(r1b, r1b + nr1);
            signalled0 = signalled = true;
          }
          // the block's rows of h are complete when all nu1 GEMM-1 units of the block have been counted in
          if (tid == 0) {
            int spins = 0;
            // (polled gently, and every block's counter in a cache line of its own: a few hundred workgroups polling
            // one line at full speed slow down every stream that crosses that memory channel)
            while (__hip_atomic_load(&p.sync[2 + blk * kDecBlockStride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < nu1) {
              __builtin_amdgcn_s_sleep(16);
              if (++spins > p.spin_limit) {
                atomicOr(&p.sync[1], 1);
                break;
              }
            }
          }
          __syncthreads();
          if (i == n1) DEC_STAMP(5);
          x_request(std::integral_constant<int, 2>{}, cur);
        } else {
          x_request(std::integral_constant<int, 1>{}, cur);
        }
        x_settle();
      }
      if (i == 0) DEC_STAMP(14);
      const int F = cur.frag;
      // ---- this wave's stages of the unit; the next unit's blocks follow into the slots as they fall free ----
      typename FR::acc_t acc[FPU][2];
#pragma unroll
      for (int f = 0; f < FPU; ++f)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[f][g][c] = 0.f;
      const int nst_next = unit_nst(nxt), nfr_next = unit_nfr(nxt);
#pragma unroll
      for (int j = 0; j < XS; ++j) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const bf16x8_t xf = __builtin_bit_cast(bf16x8_t, xr[j][t]);
#pragma unroll
          for (int f = 0; f < FPU; ++f)
#pragma unroll
            for (int g = 0; g < 2; ++g) {
              const u32x4_t v = wr[H][j][f][g];
              const uint32_t raw = t == 0 ? v.x : t == 1 ? v.y : t == 2 ? v.z : v.w;
              acc[f][g] = FR::mma(dequant8(raw, bits_f32(((sr[H][j][f][g] >> (8 * kg)) & 0xFFu) << 23)), xf, acc[f][g]);
            }
        }
        load_w(h_c, j, nxt, nst_next, nfr_next);
      }
      // ---- the waves' sums meet in LDS; half of the waves, the other half in the next unit, add two of a fragment's 16 x 32 results a lane in the waves' order and
      // finish them (one wave for all of them held up the others' next unit where units are short; all waves: themselves where they are long) ----
      if (i == 0) DEC_STAMP(15);
      DEC_UNIT_STAMP(i);
#pragma unroll
      for (int f = 0; f < FPU; ++f)
#pragma unroll
        for (int g = 0; g < 2; ++g) *reinterpret_cast<f32x4_t*>(&red_s[i & 1][wave][lr][f * 32 + ((g * 4 + kg) ^ (lr & 7)) * 4]) = acc[f][g];
      __syncthreads();
      if (i == 0) DEC_STAMP(16);
      if (i == nr0 && !signalled0) {  // the first unit behind run 0 (it exists and opened a new row block)
        signalled0 = true;
        signal_blocks(r0b, r0b + nr0);
      }
      if (i == n1 && !signalled) {  // the first GEMM-2 unit
        signalled = true;
        signal_blocks(r1b, r1b + nr1);
      }
      if ((wave & 1) == (i & 1)) {
        const int r = (wave >> 1) * 4 + (lane >> 4), c = (lane & 15) * 2;
        const int flat = rowflat_s[row0 + (r < rows ? r : rows - 1)];
        const float gam = gate_s[flat];
        // One store for either GEMM, of two bf16 results: of y (flat row t*k + j) the gate-weighted columns c and c + 1; of h (row row0 + r), by every
        // second lane, its and its neighbour's swiglu over the (gate, linear) pair
#pragma unroll
        for (int f = 0; f < FPU; ++f) {
          f32x2_t s = {0.f, 0.f};
#pragma unroll
          for (int q = 0; q < NW; ++q) s += *reinterpret_cast<const f32x2_t*>(&red_s[i & 1][q][r][f * 32 + ((c >> 2) ^ (r & 7)) * 4 + (c & 3)]);
          s += *reinterpret_cast<const f32x2_t*>(&bias_s[i][f * 32 + c]);
          const float o = swiglu_f(s[0], s[1], nalpha_log2e, limit);
          const float right = quad_swap<0xB1>(o);  // lanes 1 0 3 2 of four
          const int n = (F + f) * 32 + c;
          const bool up = ph == 1, mine = r < rows && n < (up ? p.N1 : p.N2) && !(up && (lane & 1));
          const uint32_t off = up ? (uint32_t)(row0 + r) * (uint32_t)(p.K2 * 2) + (uint32_t)n : (uint32_t)flat * (uint32_t)(p.N2 * 2) + (uint32_t)n * 2u;
          __builtin_amdgcn_raw_buffer_store_b32(up ? pack_bf16x2(o, right) : pack_bf16x2(s[0] * gam, s[1] * gam), up ? hrsrc : yrsrc, mine ? off : kDroppedStore, 0, kThrough);
        }
      }
    };
    // Whole rounds of RD units run without a test between the units: with one, the compiler has to allow for a round
    // that skips its later units and comes back to the first, i.e. for weight blocks that nothing younger follows, and
    // its waits then drain the wave's memory queue once per round.
    int i_unit = 0;
    for (; i_unit + RD <= n_units; i_unit += RD)
      static_for<0, RD>([&](auto h_c) __attribute__((always_inline)) { unit_body(h_c, i_unit + decltype(h_c)::value); });
    static_for<0, RD - 1>([&](auto h_c) __attribute__((always_inline)) {
      if (i_unit + decltype(h_c)::value < n_units) unit_body(h_c, i_unit + decltype(h_c)::value);
    });
  };  // stream
  if constexpr (FETCH != kFetchEither) {
    stream(template_int<FETCH>{});
  } else {
    const int again = nblk - A;
    // (plain loads first: they are for layers whose few experts take all tokens, the shortest ones, and the copy that stands first starts 0.6 to 1.5 us sooner.  Last / first, 60
    // tokens, 64 experts, top 4, nearly all on the same ones, 2304 56.0 / 55.2, 3072 74.0 / 72.2; 64 tokens, 128, 2880 77.5 / 76.8)
    const bool large = A * (p.nfr1 * p.nst1 + p.nfr2 * p.nst2) > kLargeBlocks;
    if (!large || again * (XS == 3 ? 3 : 10) > nblk)
      stream(template_int<kFetchPlain>{});
    else if (XS < 3 || again * 20 <= nblk)
      stream(template_int<kFetchOnce>{});
    else
      stream(template_int<kFetchEither>{});
  }
  DEC_STAMP(6);
  // ---- 4./5. hand-over of whatever is still to be counted in, then the combine of this workgroup's rows of y ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (!signalled0) signal_blocks(r0b, r0b + nr0);
  if (!signalled) signal_blocks(r1b, r1b + nr1);
  DEC_STAMP(7);
  int32_t* arrivals = p.sync + 2 + kDecBlockWords;
  const bool out_vec = (p.out_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
  for (int it0 = 0; it0 < n2 * (64 * FPU); it0 += NT) {
    // item = (unit, its fragment, row of its block, group of 8 columns): the group-0 thread counts the row in and tells the other three
    const int it = it0 + tid;
    int seen = -1, token = 0, F = 0;
    if (it < n2 * (64 * FPU)) {
      const DecUnit u = tab_s[n1 + it / (64 * FPU)];
      const int r = (it >> 2) & 15;
      const int a = (u.key >> 8) & 0xFFFF, rb = u.key & 0xFF;
      const int e = act_s[a];
      F = u.frag + (FPU == 1 ? 0 : (it >> 6) % FPU);
      if (rb * 16 + r < hist_s[e] && (FPU == 1 || F < p.nfr2)) {
        token = rowflat_s[offs_s[e] + rb * 16 + r] / k;
        if ((it & 3) == 0) seen = __hip_atomic_fetch_add(&arrivals[token * p.nfr2 + F], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    seen = __shfl(seen, lane & ~3);
    const int n0 = F * 32 + (it & 3) * 8;
    const bool sum_it = seen == k - 1 && n0 < p.N2;
    // all k rows of (token, fragment) are in memory: fp32 sum in j order, bf16 result
    const bool full = n0 + 8 <= p.N2;  // else four columns (N2 is a multiple of 4... of 8 here)
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < k; j0 += 4) {
      u32x4_t v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t off = (sum_it && j0 + q < k) ? (uint32_t)(token * k + j0 + q) * (uint32_t)(p.N2 * 2) + (uint32_t)n0 * 2u : kDroppedStore;
        v[q] = __builtin_amdgcn_raw_buffer_load_b128(yrsrc, off, 0, kThrough);  // dropped offsets read zero
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          sum[2 * c] += bits_f32(v[q][c] << 16);
          sum[2 * c + 1] += bits_f32(v[q][c] & 0xFFFF0000u);
        }
    }
    if (sum_it) {
      uint16_t* o = p.out + (int64_t)token * p.out_stride + n0;
      if (full && out_vec) {
        *reinterpret_cast<u32x4_t*>(o) = u32x4_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3]), pack_bf16x2(sum[4], sum[5]), pack_bf16x2(sum[6], sum[7])};
      } else {
        const int nc = p.N2 - n0 < 8 ? p.N2 - n0 : 8;
        for (int c = 0; c < nc; ++c) o[c] = f32_to_bf16_bits(sum[c]);
      }
    }
  }
  // ---- 6. the last workgroup to finish clears the counters for the next launch ----
  __syncthreads();
  DEC_STAMP(8);
#ifdef TK_DEC_STAMPS
  if (tid == 0) { dec_stamps[blockIdx.x][10] = n1; dec_stamps[blockIdx.x][11] = n2; }
#endif
  if (tid == 0) {
    __threadfence();
    misc_s[1] = atomicAdd(&p.sync[0], 1);
  }
  __syncthreads();
  if (misc_s[1] == G - 1) {
    __threadfence();
    for (int b = tid; b < nblk; b += NT) __hip_atomic_store(&p.sync[2 + b * kDecBlockStride], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int w = tid; w < T * p.nfr2; w += NT) __hip_atomic_store(&arrivals[w], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid == 0) __hip_atomic_store(&p.sync[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// workgroups of the kernel that are resident together on the current device (cached per device and variant)
template <int VPL, int XS, int FPU, int FETCH>
int resident_workgroups() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(moe_decode_layer_kernel<VPL, XS, FPU, FETCH>), kDecNW * 64, 0) != hipSuccess || per_cu <= 0)
      return 0;
    per_cu = 1;  // (more than half of a CU's LDS a workgroup)
    n = per_cu * device_cu_count();
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Units of one workgroup: at most min(E, R) + R / 16 row blocks, dealt evenly (+1 per run)
bool units_fit(const DecodeParams& p, int64_t units_of_block, int grid, int max_units) {
  const int64_t R = (int64_t)p.T * p.k, max_blocks = (R < p.E ? R : p.E) + R / 16;
  return max_blocks * units_of_block / grid + 4 <= max_units;
}

template <int VPL, int XS, int FPU, int FETCH>
int32_t launch_layer(const DecodeParams& p, hipStream_t st) {
  typedef DecCfg<XS, FPU> C;
  const int grid = resident_workgroups<VPL, XS, FPU, FETCH>();
  if (grid <= 0) return fail(TK_ERR_LAUNCH, "tk_moe_decode_layer: cannot determine how many workgroups are resident together");
  if (!units_fit(p, cdiv(p.nfr1, FPU) + cdiv(p.nfr2, FPU), grid, C::UNITS)) {
    if constexpr (FPU > 1) return launch_layer<VPL, kDecXS, 1, FETCH>(p, st);
    return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: row blocks of %d x %d rows x %d fragments over %d workgroups exceed the kernel's unit table", p.T, p.k, p.nfr1 + p.nfr2, grid);
  }
  hipLaunchKernelGGL((moe_decode_layer_kernel<VPL, XS, FPU, FETCH>), dim3((unsigned)grid), dim3(kDecNW * 64), 0, st, p);
  return check_launch("moe_decode_layer_kernel");
}

// K of up to 8 stages: one a wave, two fragments a unit; up to 16: two, and two fragments where there are some twenty units of one a workgroup (with fewer the
// last ones are too long).  us, stages of three a wave and one fragment a unit / two stages and one / two and two: 60 tokens, 96 experts, top 4, 2048 136 / 123 /
// 116, 16 experts 48.3 / 46.4 / 49.2; 20 tokens, 32 experts, top 2, 1600 39.5 / 36.6 / 38.1.  One stage and two fragments: 100 tokens, 64 experts, top 2, 1024 58 -> 46; 12 tokens, 32 experts,
// top 8, 1024 40 -> 31.
template <int VPL, int FETCH>
int32_t launch_layer(const DecodeParams& p, hipStream_t st) {
  const int nst = p.nst1 > p.nst2 ? p.nst1 : p.nst2, R = p.T * p.k;
  const bool two = (int64_t)(R < p.E ? R : p.E) * (p.nfr1 + p.nfr2) >= 20 * device_cu_count();
  if (nst <= kDecNW) return launch_layer<VPL, 1, 2, FETCH>(p, st);
  if (nst <= 2 * kDecNW) return two ? launch_layer<VPL, 2, 2, FETCH>(p, st) : launch_layer<VPL, 2, 1, FETCH>(p, st);
  return launch_layer<VPL, kDecXS, 1, FETCH>(p, st);
}

template <int VPL>
int32_t launch_layer(const DecodeParams& p, hipStream_t st) {
  const int fetch = decode_fetch(p.T, p.k, p.E, p.nfr1 * p.nst1 + p.nfr2 * p.nst2);
  if (fetch == kFetchPlain) return launch_layer<VPL, kFetchPlain>(p, st);
  return fetch == kFetchOnce ? launch_layer<VPL, kFetchOnce>(p, st) : launch_layer<VPL, kFetchEither>(p, st);
}

}  // namespace
}  // namespace tk

using namespace tk;

#ifdef TK_DEC_STAMPS
extern "C" int32_t tk_debug_dec_stamps(long long* host_out) {
  return hipMemcpyFromSymbol(host_out, HIP_SYMBOL(dec_stamps), sizeof(long long) * 1024 * 20) == hipSuccess ? 0 : 3;
}
#endif

extern "C" int64_t tk_moe_decode_layer_workspace_bytes(int32_t n_tokens, int32_t k, int32_t n_experts, int32_t d_ff, int32_t d_model) {
  if (n_tokens <= 0 || k <= 0 || n_experts <= 0 || d_ff <= 0 || d_model <= 0) return 0;
  const int64_t R = (int64_t)n_tokens * k;
  const int64_t hb = (R * d_ff * 2 + 255) / 256 * 256, yb = (R * d_model * 2 + 255) / 256 * 256;
  return hb + yb + (2 + (int64_t)kDecBlockWords + (int64_t)n_tokens * cdiv(d_model, 32)) * 4;
}

extern "C" int32_t tk_moe_decode_layer(const tk_decode_layer_desc* d, tk_stream_t stream) {
  if (!d) return fail(TK_ERR_INVALID, "tk_moe_decode_layer: null descriptor");
  const int T = d->n_tokens, E = d->n_experts, k = d->k;
  if (T < 0 || E <= 0 || k <= 0 || d->d_model <= 0 || d->d_ff <= 0) return fail(TK_ERR_INVALID, "tk_moe_decode_layer: bad sizes T=%d E=%d k=%d d_model=%d d_ff=%d", T, E, k, d->d_model, d->d_ff);
  if (T == 0) return TK_OK;
  if (k > E || k > 32) return fail(TK_ERR_INVALID, "tk_moe_decode_layer: k=%d must be <= min(32, E)", k);
  if ((int64_t)T * k > kDecMaxRows) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: at most %d routed rows (got %d x %d); larger batches take tk_route + tk_moe_gemm", kDecMaxRows, T, k);
  if (E > kDecMaxExperts) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: at most %d experts (got %d)", kDecMaxExperts, E);
  const int kmax = kDecNW * kDecXS * 128;
  if (d->d_model > kmax || d->d_ff > kmax) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: d_model and d_ff must be <= %d (got %d, %d)", kmax, d->d_model, d->d_ff);
  if (d->d_model % 8 || d->d_ff % 8) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: d_model and d_ff must be multiples of 8 (got %d, %d)", d->d_model, d->d_ff);
  if (!d->x || !d->logits || !d->w1 || !d->w1_mx_scale || !d->w2 || !d->w2_mx_scale || !d->out || !d->workspace) return fail(TK_ERR_INVALID, "tk_moe_decode_layer: null operand");
  if (d->logits_dtype != TK_F32 && d->logits_dtype != TK_BF16) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: logits must be fp32 or bf16");
  if ((d->b1 && d->b1_dtype != TK_F32 && d->b1_dtype != TK_BF16) || (d->b2 && d->b2_dtype != TK_F32 && d->b2_dtype != TK_BF16)) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: biases must be fp32 or bf16");
  if ((reinterpret_cast<uintptr_t>(d->x) & 15) || d->x_stride_m % 8) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: activation rows must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(d->workspace) & 255)) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: the workspace must be 256-byte aligned");
  for (const void* q : {d->w1, d->w2})
    if (reinterpret_cast<uintptr_t>(q) & 15) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: tiled weights must be 16-byte aligned");
  for (const void* q : {d->w1_mx_scale, d->w2_mx_scale})
    if (reinterpret_cast<uintptr_t>(q) & 3) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: tiled scales must be 4-byte aligned");
  DecodeParams p;
  p.x = static_cast<const uint8_t*>(d->x);
  p.x_stride = d->x_stride_m;
  {
    const int64_t extent = ((int64_t)(T - 1) * d->x_stride_m + d->d_model) * 2;
    if (d->x_stride_m < d->d_model || extent > 0x7FFFFFFFll) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: activation rows must not overlap and must lie within 2 GiB (row stride %lld)", (long long)d->x_stride_m);
    p.x_bytes = (uint32_t)extent;
  }
  p.logits = d->logits;
  p.logits_stride = d->logits_stride_m;
  p.logits_is_bf16 = d->logits_dtype == TK_BF16;
  p.T = T;
  p.E = E;
  p.k = k;
  p.apply_softmax = d->apply_softmax;
  p.K1 = d->d_model;
  p.N1 = 2 * d->d_ff;
  p.K2 = d->d_ff;
  p.N2 = d->d_model;
  p.nst1 = (int)cdiv(p.K1, 128);
  p.nst2 = (int)cdiv(p.K2, 128);
  p.nfr1 = (int)cdiv(p.N1, 32);
  p.nfr2 = (int)cdiv(p.N2, 32);
  if (d->w1_stride_e % 16 || d->w2_stride_e % 16 || d->w1s_stride_e % 4 || d->w2s_stride_e % 4) return fail(TK_ERR_UNSUPPORTED, "tk_moe_decode_layer: expert strides of tiled weights must be multiples of 16 (scales: 4) bytes");
  if (E > 1 && (d->w1_stride_e < (int64_t)p.nfr1 * p.nst1 * 2048 || d->w1s_stride_e < (int64_t)p.nfr1 * p.nst1 * 128 ||
                d->w2_stride_e < (int64_t)p.nfr2 * p.nst2 * 2048 || d->w2s_stride_e < (int64_t)p.nfr2 * p.nst2 * 128))
    return fail(TK_ERR_INVALID, "tk_moe_decode_layer: expert stride smaller than one tiled expert");
  p.w1 = static_cast<const uint8_t*>(d->w1);
  p.w1s = static_cast<const uint8_t*>(d->w1_mx_scale);
  p.w1_stride_e = d->w1_stride_e;
  p.w1s_stride_e = d->w1s_stride_e;
  p.b1 = d->b1;
  p.b1_stride_e = d->b1_stride_e;
  p.b1_is_f32 = d->b1_dtype == TK_F32;
  p.w2 = static_cast<const uint8_t*>(d->w2);
  p.w2s = static_cast<const uint8_t*>(d->w2_mx_scale);
  p.w2_stride_e = d->w2_stride_e;
  p.w2s_stride_e = d->w2s_stride_e;
  p.b2 = d->b2;
  p.b2_stride_e = d->b2_stride_e;
  p.b2_is_f32 = d->b2_dtype == TK_F32;
  p.alpha = d->act_alpha;
  p.limit = d->act_limit;
  p.has_limit = d->act_has_limit;
  const int64_t R = (int64_t)T * k;
  const int64_t hb = (R * p.K2 * 2 + 255) / 256 * 256, yb = (R * p.N2 * 2 + 255) / 256 * 256;
  uint8_t* ws = static_cast<uint8_t*>(d->workspace);
  p.h = reinterpret_cast<uint16_t*>(ws);
  p.y = reinterpret_cast<uint16_t*>(ws + hb);
  p.sync = reinterpret_cast<int32_t*>(ws + hb + yb);
  p.out = static_cast<uint16_t*>(d->out);
  p.out_stride = d->out_stride_m;
  p.indx_out = static_cast<int16_t*>(d->indx_out);
  p.vals_out = d->vals_out;
  p.spin_limit = d->spin_limit > 0 ? d->spin_limit : (1 << 22);
  if (d->spin_limit <= 0 && decode_by_rows(T, k, d->d_ff, d->d_model)) return decode_launch_rows(p, static_cast<hipStream_t>(stream));
  hipStream_t st = static_cast<hipStream_t>(stream);
  return E <= 128 ? launch_layer<8>(p, st) : launch_layer<kDecMaxExperts / 16>(p, st);
}
