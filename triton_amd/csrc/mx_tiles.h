// How the MX kernels for a strided axis (mx_quant.hip) cut a 16-bit tensor [outer, L, inner] into tiles of 256 columns.  Plain C++: a launch takes the
// number of workgroups and the kernel (the blocks of 32 in a tile, how the source is read) from the same answer.
#pragma once
#include <stdint.h>

namespace tk {

constexpr int kMxTileCols = 256;
constexpr int kMxSmallBlocks = 4;                                                  // blocks of a small tile: one a wave
constexpr int mx_tile_blocks(bool e2m1) { return e2m1 ? 8 : 4; }                   // ... of one whose columns are whole lines of 128 bytes

// e2m1: small tiles, one block a wave instead of two, where those of whole lines are up to four a CU (up: two): both directions are a chain of loads, conversion and stores, and
// half of it is shorter (us, both launches: 1 x 2368 x 592 14.6 -> 9.7, 11 x 448 x 256 14.3 -> 9.4, 5 x 544 x 2368 15.9 -> 11.6, 8 x 1024 x 1024 15.3 -> 12.5, 1 x 2880 x 5760 (276 tiles)
// 24.5 -> 20.3, 2 x (552) 35.1 -> 32.8, 16 x 2048 x 1024 (512) 30.8 -> 29.3; 8 x 2880 x 2880 (1152) 65.1 -> 66.6, since a column's piece is half a line).
// Up, other tensors in turn, whole-line / small tiles: 2 x 2880 x 2880 (276) 15.1 / 12.2, 3 x (414) 16.7 / 15.0, 8 x 2048 x 2048 (512) 20.8 / 20.5, 2 x 2880 x 5760 (552) 20.5 / 22.1, 3 x
// (828) 27.0 / 29.3: half lines are fetched twice where nothing of the tensor is in a cache.
constexpr int64_t kMxSmallTiles = 1024, kMxSmallTilesUp = 512;

// Sources of this size and more are read with the non-temporal hint; to e2m1, whose values are a quarter of the source, from less on where the rows begin at multiples of 8
// bytes.  What the program wrote or read a moment ago is in the memory-side cache up to about a hundred megabytes, and a read with the hint does not profit from that;
// what it did not touch lately, as a first call on loaded weights has it, is read faster with the hint.  us a launch, plain loads / with the hint: the same tensor again and
// again; others in turn; one that the kernel in front has just made.  bf16 to e2m1, small tiles:
//   8 x 1024 x 1024 (17 MB) 4.7 / 4.7; 7.3 / 6.7; 9.6 / 13.0; 2 x 2880 x 2880 (33 MB) 9.0 / 10.7; 13.7 / 12.4; 11.7 / 12.0; 3 x (50 MB) 13.2 / 13.9; 18.3 / 15.7; 13.6 / 16.6
//   8 x 2048 x 2048 (67 MB) 15.6 / 18.4; 22.7 / 20.1; 16.5 / 19.1; 2 x 2880 x 5760 (66 MB) 16.6 / 18.8; 22.3 / 19.8; 16.5 / 17.1; 3 x (100 MB) 22.1 / 27.1; 30.3 / 27.6; 21.7 / 27.1
//   (whole-line tiles with the hint, as all sizes had them once, 33 MB 11.9; 13.6; 14.3; 50 MB 14.1; 15.5; 15.9; 100 MB 28.3; 28.9; 27.4)
//   rows at any address, 16 x 2048 x 1093 (72 MB) 17.1 / 22.7; 24.4 / 22.7; 17.6 / 23.1
// To e4m3: 3 x 2880 x 2880 15.5 / 18.1; 21.2 / 18.9; 15.1 / 18.3; 2 x 2880 x 5760 18.9 / 24.8; 26.6 / 24.7; 18.6 / 18.7; 3 x 25.5 / 34.0; 36.3 / 33.8; 24.6 / 32.4; 4 x (133 MB) 35.2 / 43.9;
//   47.2 / 43.7; 37.2 / 46.6; two in turn: 4 x 47.8 / 39.5, 8 x 107 / 75, 16 x 181 / 153, 32 x 343 / 300.
constexpr int64_t kMxOnceBytes = 96ll << 20, kMxOnceBytesE2m1 = 36ll << 20;

// Up: a tile's bytes requested together up to this many (small) tiles, two a CU.  us, one piece after the other / together, the same tensor again and again; others in turn:
//   from e2m1: 960 x 517 (24 tiles) 4.1 / 3.8; 5.2 / 4.3; 2 x 1024 x 517 (48) 4.4 / 4.0; 6.2 / 4.7; 8 x 1024 x 1024 (256) 6.2 / 5.9; 8.7 / 7.3; 4 x 2048 x 2048 (512) 9.9 / 9.3; 11.7 / 11.2;
//   2 x 2880 x 2880 (552) 10.5 / 10.9; 12.2 / 13.2; 3 x (828) 13.6 / 14.2; 15.1 / 17.1
//   from e4m3: 960 x 517 5.0 / 4.5; 6.8 / 4.9; 2 x 1024 x 517 5.3 / 4.7; 8.9 / 5.8 (7.2 by a column a lane, which calls of that kind took once); 2880 x 517 (69) 5.7 / 5.0; 9.6 / 6.6 (7.9);
//   8 x 1024 x 1024 7.0 / 6.3; 11.3 / 8.7; 4 x 2048 x 2048 11.6 / 10.3; 15.8 / 14.4; 2 x 2880 x 2880 12.1 / 11.4; 15.1 / 16.9; 8 x 2048 x 2048 (1024) 21.7 / 20.0; 25.9 / 28.4
constexpr int64_t kMxTogether = 512;

struct MxTiles {
  int64_t col_tiles, blk_tiles, grid;
  int32_t blocks;  // of 32, in a tile
  bool once;       // down: the source is read with the non-temporal hint
  bool together;   // up: a tile's bytes are requested together
};

// down: a source to be quantised, rows8: its rows begin at multiples of 8 bytes
inline MxTiles mx_tiles(int64_t outer, int64_t L, int64_t inner, bool e2m1, bool down, bool rows8) {
  const int64_t nblk = L / 32;
  MxTiles t;
  t.col_tiles = (inner + kMxTileCols - 1) / kMxTileCols;
  t.blocks = mx_tile_blocks(e2m1);
  t.once = down && outer * L * inner * 2 >= (e2m1 && rows8 ? kMxOnceBytesE2m1 : kMxOnceBytes);
  if (t.col_tiles * ((nblk + t.blocks - 1) / t.blocks) * outer <= (down ? kMxSmallTiles : kMxSmallTilesUp)) t.blocks = kMxSmallBlocks;
  t.blk_tiles = (nblk + t.blocks - 1) / t.blocks;
  t.grid = t.col_tiles * t.blk_tiles * outer;
  t.together = !down && t.blocks == kMxSmallBlocks && t.grid <= kMxTogether;
  return t;
}

// Whether a source whose rows begin at any address (an odd number of columns, say) is quantised by a column a lane instead: up to some 70 tiles that kernel's shorter chain is the
// faster one.  us, bf16, by tiles / by columns, the same tensor again and again; others in turn: to e2m1, 480 x 1093 (20 tiles) 5.0 / 4.4 (others), 960 x 517 (24) 5.9 / 3.8; 6.0 / 4.4, 960 x 1093
// (40) 4.5 / 3.8; 5.5 / 5.2, 2 x 1024 x 517 (48) 5.7 / 4.0; 6.0 / 5.0, 2880 x 517 (69) 5.6 / 4.3; 6.4 / 6.0, 480 x 4097 (68) 4.6 / 4.4; 6.3 / 6.4, 4 x 960 x 517 (96) 4.6 / 5.1; 6.3 / 6.7, 2880 x 1093 (115) 4.8 /
// 4.8; 6.8 / 7.3; to e4m3, 960 x 517 6.1 / 4.0; 6.2 / 4.6, 4 x 960 x 517 5.2 / 4.8; 7.0 / 6.9, 2880 x 1093 5.6 / 5.6; 7.5 / 7.6.
// Except where the last of its 64 columns are one to eight and the launch is small, which then takes 5.5 to 6.5 (a tile with as few columns takes as long): 480 x 65 4.1 / 5.8, 960 x 193 4.5 / 6.1, 480 x 897
// (60 workgroups) 5.0 / 5.4, 960 x 577 (80) 5.0 / 4.4.
inline bool mx_by_columns(int64_t outer, int64_t L, int64_t inner) {
  const int64_t quads = (L / 32 + 3) / 4 * outer, last = inner % 64;
  if ((inner + kMxTileCols - 1) / kMxTileCols * quads > 70) return false;
  return !(last >= 1 && last <= 8 && inner % kMxTileCols > 8 && (inner + 63) / 64 * quads < 64);
}

}  // namespace tk
