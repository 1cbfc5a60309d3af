// How the MX kernels for a strided axis (mx_quant.hip) cut a 16-bit tensor [outer, L, inner] into tiles of 256 columns.  Plain C++: a launch takes the
// number of workgroups and the kernel (the blocks of 32 in a tile, how the source is read) from the same answer.
#pragma once
#include <stdint.h>

namespace tk {

constexpr int kMxTileCols = 256;
constexpr int kMxSmallBlocks = 4;                                                  // blocks of a small tile: one a wave
constexpr int mx_tile_blocks(bool e2m1) { return e2m1 ? 8 : 4; }                   // ... of one whose columns are whole lines of 128 bytes

// e2m1: small tiles, one block a wave instead of two, where those of whole lines are up to four a CU: both directions are a chain of loads, conversion and stores, and
// half of it is shorter (us, both launches: 1 x 2368 x 592 14.6 -> 9.7, 11 x 448 x 256 14.3 -> 9.4, 5 x 544 x 2368 15.9 -> 11.6, 8 x 1024 x 1024 15.3 -> 12.5, 1 x 2880 x 5760 (276 tiles)
// 24.5 -> 20.3, 2 x (552) 35.1 -> 32.8, 16 x 2048 x 1024 (512) 30.8 -> 29.3; 8 x 2880 x 2880 (1152) 65.1 -> 66.6, since a column's piece is half a line).
constexpr int64_t kMxSmallTiles = 1024;

// Sources of this size and more are read with the non-temporal hint, by whole-line tiles.  Two in turn, plain loads / with the hint, us a launch, bf16 [b, 2880, 5760] to e4m3:
// b 2 (66 MB) 18.1 / 23.8, b 4 47.8 / 39.5, b 8 107 / 75, b 16 181 / 153, b 32 343 / 300; to e2m1: b 2 18.9 / 21.8, b 4 42.6 / 36.8, b 8 95 / 68.  What
// was used a moment ago is still in the memory-side cache up to about a hundred megabytes, and a read with the hint does not profit from that.
constexpr int64_t kMxOnceBytes = 96ll << 20;

struct MxTiles {
  int64_t col_tiles, blk_tiles, grid;
  int32_t blocks;  // of 32, in a tile
  bool once;       // down: the source is read with the non-temporal hint
};

inline MxTiles mx_tiles(int64_t outer, int64_t L, int64_t inner, bool e2m1, bool down) {
  const int64_t nblk = L / 32;
  MxTiles t;
  t.col_tiles = (inner + kMxTileCols - 1) / kMxTileCols;
  t.blocks = mx_tile_blocks(e2m1);
  t.once = down && outer * L * inner * 2 >= kMxOnceBytes;
  if (!t.once && t.col_tiles * ((nblk + t.blocks - 1) / t.blocks) * outer <= kMxSmallTiles) t.blocks = kMxSmallBlocks;
  t.blk_tiles = (nblk + t.blocks - 1) / t.blocks;
  t.grid = t.col_tiles * t.blk_tiles * outer;
  return t;
}

}  // namespace tk
