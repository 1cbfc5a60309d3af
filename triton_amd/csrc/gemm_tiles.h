// Tiles of the persistent kernels that fetch their operands by memory-to-LDS transfers, found from the slice sizes alone.
#pragma once
#include "gemm_common.h"
#include "route_common.h"

namespace tk {
namespace {

constexpr uint32_t kOutOfRange = 0x80000000u;  // byte offset that every buffer resource here (below 2 GiB) treats as out of range
constexpr int kSliceRegs = kDmaSlices / 64;

struct Tile {
  int expert, off_m, start_m, eM, n_tile;
  bool narrow;
};

// Two lists: row blocks that are more than half full, then the short last blocks of the experts, which cost a fraction of a tile;
// with the short ones in between, a workgroup's share was up to a whole tile longer than the next one's.  Of each list every
// XCD (workgroup b runs on XCD b % 8) takes a contiguous part, walked side by side by its workgroups, the short tiles behind the
// others: the workgroups without a tile in the last round of full ones begin with them.
// Slice sizes and offsets stay in registers, lane l of register c holding slice c * 64 + l.
// SBN < BN: short row blocks may be cut into tiles of SBN columns instead ("narrow"): where those of the whole width neither find room beside the
// last full tiles nor keep more than half of the workgroups busy behind them.  (256 workgroups, K 2048, N 4096: 256 full and 112 short
// tiles 95.5 -> 85 us; 128 full and 128 short tiles, which are one round, 47 against 59 in narrow ones.)
template <int BM, int BN, int SBN = BN>
struct TileList {
  int sz[kSliceRegs], so[kSliceRegs];
  int f_beg, f_len, s_beg, t_end, t_step, grid_n;
  int grid_s = 0;  // SBN < BN: tiles of a short row block if those are narrow, else 0

  static __device__ __forceinline__ int n_full(int rows) { return (rows + BM / 2 - 1) / BM; }
  static __device__ __forceinline__ int n_short(int rows) { return rows > n_full(rows) * BM ? 1 : 0; }

  // n_cols = tiles of a row block; returns this workgroup's first index (it has none if that is not below t_end; the following ones are t_step apart)
  __device__ __forceinline__ int init(const GemmParams& p, int lane, int n_cols) {
    int full = 0, brief = 0;
#pragma unroll
    for (int c = 0; c < kSliceRegs; ++c) {
      const int e = c * 64 + lane;
      sz[c] = so[c] = 0;
      if (p.slice_sizes) {
        if (e < p.n_slices) {
          sz[c] = p.slice_sizes[e];
          so[c] = p.slice_offs[e];
        }
      } else if (e == 0) {
        sz[c] = p.M;
      }
    }
#pragma unroll
    for (int c = 0; c < kSliceRegs; ++c) {
      full += __builtin_amdgcn_readlane(wave_scan_i32(n_full(sz[c])), 63);
      brief += __builtin_amdgcn_readlane(wave_scan_i32(n_short(sz[c])), 63);
    }
    grid_n = n_cols;
    if constexpr (SBN < BN) {
      const uint32_t wgs = gridDim.x, over = (uint32_t)(full * grid_n) % wgs, wide = (uint32_t)(brief * grid_n);
      if (wide > (over ? wgs - over : 0) && wide * 2 <= wgs) grid_s = (p.N + SBN - 1) / SBN;
    }
    const int xcd = blockIdx.x & 7;
    t_step = gridDim.x >> 3;
    // An eighth of the full tiles, and of the short ones what makes an eighth of all: with each list divided on its own an XCD could be two
    // tiles over, which one workgroup then had in a round of its own (94 rows a slice, three rounds, K 2880, N 2880: 195 -> 169 us).
    // (From eight short tiles on their bounds only grow: an eighth of all is then at least the larger eighth of the full ones.)
    const int64_t n_f = (int64_t)full * grid_n, n_s = (int64_t)brief * (grid_s ? grid_s : grid_n), n = n_f + n_s;
    auto full_to = [&](int x) -> int { return (int)((n_f * x) >> 3); };
    auto short_to = [&](int x) -> int { return n_s < 8 ? (int)((n_s * x) >> 3) : (int)((n * x) >> 3) - full_to(x); };
    f_beg = full_to(xcd), f_len = full_to(xcd + 1) - f_beg;
    s_beg = short_to(xcd);
    t_end = f_len + short_to(xcd + 1) - s_beg;
    return (int)(blockIdx.x >> 3);
  }

  __device__ __forceinline__ Tile locate(int t) const {
    Tile r = {0, 0, 0, 0, 0, false};
    const bool is_full = t < f_len;
    const int g = is_full ? f_beg + t : s_beg + t - f_len;
    r.narrow = SBN < BN && !is_full && grid_s;
    const int grid_n = r.narrow ? grid_s : this->grid_n;
    const int q = g / grid_n;
    int base = 0;
    bool found = false;
#pragma unroll
    for (int c = 0; c < kSliceRegs; ++c) {
      if (found) continue;
      const int cnt = is_full ? n_full(sz[c]) : n_short(sz[c]);
      const int inc = wave_scan_i32(cnt);
      const int total = __builtin_amdgcn_readlane(inc, 63);
      if (q < base + total) {
        found = true;
        const int l = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(base + inc > q));
        const int nb = __builtin_amdgcn_readlane(cnt, l);
        int i = g - (base + __builtin_amdgcn_readlane(inc, l) - nb) * grid_n;
        r.expert = c * 64 + l;
        r.eM = __builtin_amdgcn_readlane(sz[c], l);
        r.start_m = __builtin_amdgcn_readlane(so[c], l);
        // bands of eight row blocks, in a band column by column, so that the tiles an XCD has in hand share eight blocks of
        // activations and a few of weights through its L2
        const int band = i / (8 * grid_n);
        const int bh = nb - band * 8 < 8 ? nb - band * 8 : 8;
        i -= band * 8 * grid_n;
        const int pn = i / bh;
        r.n_tile = pn * (r.narrow ? SBN : BN);
        r.off_m = (is_full ? band * 8 + i - pn * bh : n_full(r.eM)) * BM;
      }
      base += total;
    }
    return r;
  }
};

}  // namespace
}  // namespace tk
