// What a call has to be like for the expert-GEMM kernels that address x through one buffer resource.  Plain C++: the entry point
// (moe_gemm.hip) picks the kernel by it and the host path (host_path.cpp, for both of its callers) the row blocks, so that row
// blocks which only such a kernel has are never chosen for a call that it cannot run.  And how a decode layer is launched: its entry
// point (moe_decode_layer.hip) and those who make its workspace go by the same rule.  And the tile of a ragged-K GEMM.
#pragma once
#include <math.h>
#include <stdint.h>

namespace tk {

// Slices whose sizes and offsets these kernels keep in registers; other kernels run with more.
constexpr int kDmaSlices = 256;

// Bytes of x for a buffer resource; 0 = x is not one: rows over 2 GiB and more, or rows that overlap (closer together than their
// length: one row expanded to many, sliding windows), whose last ones would reach past rows * stride.
inline uint32_t x_extent(int64_t rows, int64_t stride, int64_t K, int64_t itemsize) {
  const int64_t bytes = rows * stride * itemsize;
  return stride >= K && bytes > 0 && bytes < (int64_t)1 << 31 ? (uint32_t)bytes : 0u;
}

// The memory-to-LDS kernel: x as above, an expert's weights (`w_bytes`) within 2 GiB, the slices in registers.
inline bool dma_runs(uint32_t x_bytes, int64_t n_slices, int64_t w_bytes) {
  return x_bytes != 0 && n_slices <= kDmaSlices && w_bytes < (int64_t)1 << 31;
}

// ... on strided 16-bit weights, whose columns may not overlap either.
inline bool dma_runs_16bit(uint32_t x_bytes, int64_t n_slices, int64_t K, int64_t N, int64_t w_stride_n) {
  return w_stride_n >= K && dma_runs(x_bytes, n_slices, ((N - 1) * w_stride_n + K) * 2);
}

// ... on tiled e4m3 weights (fragments of 32 columns, stages of 256 k, 8 KiB each).
inline bool dma_runs_e4m3(uint32_t x_bytes, int64_t n_slices, int64_t K, int64_t N) {
  return dma_runs(x_bytes, n_slices, (N + 31) / 32 * ((K + 255) / 256) * 8192);
}

// Whether the weights (`row_bytes` a column) are fetched with the non-temporal hint: few slices have a second row block, and they are more than
// half of the 256 MiB of the cache in front of memory, so that next to nothing of them is there when the call is made again.  Measured (us of a
// layer, with against without it; other weights each call).  e4m3, 8 experts, d 4096, d_ff 14336: 8 rows each 238 against 267, 62 rows 295 / 313; d 2048, d_ff
// 4096, 16 rows (201 MB in all) 70 / 74, but with the same weights again 66 / 64.  bf16, d and d_ff 2048: 16 experts, 25 rows 112 / 120, 32 experts, 31
// rows 203 / 217; tiles of 256 rows: 32 experts, 200 rows 254 / 271; where row blocks of 256 share their weights it costs: 16 experts, 256 rows 193 / 187;
// tiles of 128 rows, 125 rows 149 / 146.  MXFP4, 128 experts, d and d_ff 2880, 128 rows 806 / 824, MXFP8 572 / 580, 94 rows 497 / 520.
// Why the line lies at 13/16 of a block (a first GEMM by itself, two sets of weights in turn, random routing): with tiles of 256 rows it turns between
// 0.85 and 0.90, where slices begin to have a second block, which the kernel without the hint cuts into narrow tiles: bf16, 32 slices, K 2048, N
// 4096: 205 rows 143 / 149, 218 144 / 150, 230 172 / 165, 243 180 / 170; 64 slices, N 1024: 218 rows 74 / 82, 230 105 / 96; e4m3, 16 slices, K 4096,
// N 8192: 218 rows 127 / 135, 230 131 / 135, 243 162 / 148 (all slices alike 3 to 14 % for the hint up to a whole block).  Smaller tiles have no
// narrow ones and gain beyond the line as well: 128 rows, 16 slices, K 2048, N 3072: 102 rows 52 / 56, 109 54 / 57, 122 53 / 57; the wide kernel's
// 160, 128 slices, K 2880, N 5760: MXFP4 128 rows 537 / 546, 136 570 / 578, 152 640 / 644, MXFP8 128 rows 358 / 357, 136 363 / 373, 152 417 / 421.  Tiles of 320
// rows, one block for a slice of 256: 32 slices, K and N 2048, 256 rows 102 / 109, N 4096 190 / 191, K 1440 163 / 152, K 2048, N 1440 92 / 100; 8 slices, K and N 4096, 256 rows 96 /
// 103; beyond the line, 285 rows, 16 slices, K 2048, N 4096 117 / 126, N 2048 58 / 65, 32 slices 123 / 127.
inline bool reads_once(int64_t rows, int64_t n_slices, int64_t block_rows, int64_t N, int64_t row_bytes) {
  const int64_t read = n_slices < rows ? n_slices : rows;
  return rows * 16 <= n_slices * block_rows * 13 && read * N * row_bytes > 128 << 20;
}

// Tile of the wide MXFP4 kernel (moe_gemm_mxw_kernel.h) for a call whose rows are more than the decode kernel is made for; rows 0 = the kernels before it.
// Figures: us, both GEMMs of a layer; "before" = the streaming kernel's 32-row blocks, or 64 and 128 rows of the ones with weights in registers.
// bf16 rows.  32 x 256 (two workgroups a CU) is the shortest chain and divides best, for one round and up to 20 rows; beyond seven rows 64 x 512, half the reads of the
// rows, where its tiles are three a CU.  Not below: there only slices with favourites fill such a tile, and they are few (real layers, the streaming
// kernel / 32 x 256 / 64 x 512; 128 slices, K 2880, random: 3 rows 277 / 268 / 275, 5 306 / 293 / 299, 8 325 / 317 / 313, 13 340 / 326 / 325, 19 368 / 341 / 339;
// with favourites, the logits' spread 1.5 times their noise: 5 rows 149 / 136 / 170, 8 192 / 189 / 177, 13 241 / 219 / 225, 19 292 / 282 / 266; all tokens on the same four: 5
// rows 70 / 64 / 87, 8 104 / 99 / 92.  K 2048: 8 rows 170 / 168 / 163, favourites 109 / 102 / 99, 16 178 / 176 / 171; 96 slices, K 1088, 12 rows 62 / 60 / 71; 64
// slices, K 1536: 9 rows 66 / 63 / 68, 19 75 / 76 / 75; 32 slices, K 2880, 19 rows 109 / 104 / 106; K 1024, N 2048, 64 slices, the first GEMM alone: 4 rows 19.0 / 18.0 /
// 17.8, favourites 11.8 / 12.5 / 18.6).  64 x 256, two workgroups a CU as well, divides a small
// product of more rows evenly; where the tiles of 512 columns are two rounds and more, those: half the reads of the rows, and three stages of weights in flight.
//   128 slices, K 2880, N 5760 and 2880: 28 rows before 415, 370 (64 x 512), 42 471, 416, 56 525, 475 (96; 64 x 512 498), 72 607, 544 (96; 160 563,
//   64 x 256 743), 84 646, 602 (160; 96 613)
//   128 slices, K 2048, N 4096: 28 rows 131, 117 (64 x 512; 64 x 256 123), 69 203, 177 (96), 109 271, 236 (160; 64 x 256 268)
//   96 slices, K 1088 and 1024, N 2048 and 1088: 39 rows 76, 60 (64 x 256; 64 x 512 72), 62 91, 74 (96 89, 160 98), 94 105, 90
//   64 slices, K 1344 and 992, N 1984 and 1344: 44 rows 68, 54, 62 80, 66, 94 93, 76 (160: 78)
//   32 slices, K 1536 and 640, N 1280 and 1536: 16 rows 32, 25 (32; 64 x 256 28), 64 46, 32 (32 or 64 x 256), 82 51, 37
//   32 slices, K 1024, N 4096: 62 rows 32, 29 (64 x 256), 500 163, 134 (160; 64 x 256 145); 16 slices, K 1024, N 2048: 50 rows 18.6, 13.1 (32; 64 x
//   256 15.1), 375 45, 34 (64 x 256)
//   (Against: products of one round with a random routing, one GEMM: 32 slices, K 2400, N 1920, 31 rows 23.7, 24.9, 16 slices, K 1024, N 4096, 37 rows 15.9, 16.9; with
//   favourites 37.6, 24.8 and 31.4, 16.5; the whole layers 101, 54 and 56, 42.)
// MXFP8 rows, whose stage is half as long to multiply: the kernel before (128 x 256 tiles, weights in registers) stays where its tiles are one round (32
// slices, K 2400, N 1920: 18 rows 21 against 24, 50 22 against 30).  Beyond that tiles as high as a routing with favourites needs as well, since the epilogue
// costs by rows: 128 x 512 from 40 rows, 64 x 512 below (whole layers, 64 / 128 rows, random and with favourites: 128 slices of 2880, 25 rows 324 / 355 and 265 / 263, 31 340 /
// 371 and 292 / 296, 37 353 / 386 and 303 / 329, 44 382 / 394 and 339 / 333, 50 412 / 404 and 366 / 361; of 1408, 26 rows 107 / 122 and 99 / 94, 32 112 / 128 and 100 / 108; 64 slices of 2048, 36
// rows 105 / 110 and 107 / 109, 44 121 / 114 and 118 / 110), and 32 x 256 up to 24 where the tiles of 512 columns are less than three a CU.
// Where these are just one round if all slices have rows, a routing with favourites makes 64-row blocks a second one from about 32 rows on (64 slices, K and N
// 2048: 37 rows, random / favourites, before 38 / 39, 64 x 512 33 / 42, 128 x 512 33 / 36; 32 slices, N 4096: 37 / 38, 32 / 42, 33 / 36; 160 tiles, K 960, N 2400: 19 /
// 21, 17 / 17, 18 / 23). 
// (All tokens on the same few experts, which a balanced router does not do, leave the tiles of 512 columns fewer than CUs, or just over a round, more often
// than the 128 x 256 ones before; layers: 128 experts of 2880, four of them live, 300 tokens 90, 83, 700 139, 162, 1400 206, 237, 2300 312, 292; 96 experts, K 1696 and 1088, 900 tokens
// 74, 78; 64 experts of 1024, two live, 300 41, 37, 1500 51, 60.)
// Before and by these rules (slices all alike; by favourites, the last one's expectation five times the first's):
//   128 slices, K 2880, N 5760 and 2880: 4 rows 348, 287 (64); 139, 135.  14 354, 305 (64); 209, 204.  28 378, 341 (128; 64 334); 262, 276 (64 289).
//   43 401, 369 (128); 322, 313 (64 357).  72 452, 418 (160 435); 427, 413.  94 485, 458 (160 467); 500, 486.  128 658, 656 (160 531); 603, 580
//   96 slices, K 1696 and 1088, N 2176 and 1696: 11 rows 92, 72 (32; 64 76); 65, 54 (64).  36 98, 86 (64; 128 90, 32 107); 88, 84 (128 96).  58 108,
//   97 (128); 106, 99.  83 121, 110; 122, 129.  125 154, 138 (160; 128 147); 153, 161 (128 144)
struct MxwTile {
  int32_t rows, cols;
};
// MXFP8 rows, more than 104 a slice: by what a tile costs.  A workgroup's tile of bm rows takes `start` + `stage` us for every 128 of K, the rounds of 256
// workgroups follow one another, and a routing makes about 1 + sum over j of P(rows > j bm) row blocks of a slice (normal, a fifth wider than random; from
// three on, half a block more than there are rows for).  How many rounds a number of tiles is near a whole one is not known: the mean of 5 % less and
// more.  The two constants of each tile come from products of one round (K 512 and 1600, 16 slices of 108 rows); the rest follows, within some 10 %: us, predicted /
// measured, 64 x 512, 128 x 512, 160 x 512, and the 128 x 256 tiles with weights in registers:
//   16 slices, K 2752, N 2368, 138 rows 30 / 31, 44 / 43, 59 / 50; K 1696, N 5440, 474 rows 114 / 115, 102 / 91, 119 / 112, 108 / 105; K 2720, N 1696 70 / 56, 64 / 65, 59 / 53, 49 / 49
//   32 slices, K 2496, N 4608, 212 rows 126 / 130, 115 / 112, 157 / 131, 108 / 115; K 2144, N 896, 494 rows 57 / 63, 69 / 58, 49 / 47; K 608, N 3968, 486 rows 81 / 87, 79 / 76, 84 / 82,
//   90 / 93; 64 slices, K 1696, N 4736, 136 rows with favourites 141 / 131, 145 / 112, 119 / 134; 128 x 256: K 640, N 3200, 32 slices of 332 54 / 65
// (160 x 512 before up to 176 rows and from 640, 128 x 256 between: 16 slices of 122 rows, K 1792, N 2048 38 -> 23; layers of 1000 tokens, 16 experts, top 8, 1536 112 -> 102, of 1500, 32
// experts, top 8, 2016 and 992 154 -> 135, of 4000, 32 experts, top 4, 2880 516 -> 473.)  Where a slice of 105 to 152 rows, one block of 160, makes three rounds of tiles
// and more, the second blocks that a routing adds are few rows each and cost less than this counts: those stay.
inline double mx8_row_blocks(double per_slice, int bm) {
  if (per_slice >= 3.0 * bm) return per_slice / bm + 0.5;
  double n = 1.0;
  const double spread = 1.2 * sqrt(per_slice);
  for (int j = 1; j < 5; ++j) n += 1.0 / (1.0 + exp(1.7 * (j * bm - per_slice) / spread));
  return n;
}
inline MxwTile mx8_tile(int64_t rows, int64_t n_slices, int64_t K, int64_t N) {
  if (rows <= 152 * n_slices && n_slices * ((N + 511) / 512) >= 3 * 256) return {160, 512};
  struct Cost {
    MxwTile tile;
    int bm, bn;
    double start, stage;
  };
  const Cost costs[] = {{{0, 0}, 128, 256, 5.1, 0.78}, {{64, 512}, 64, 512, 4.0, 1.02}, {{128, 512}, 128, 512, 7.7, 1.46}, {{160, 512}, 160, 512, 9.8, 2.05}};
  MxwTile best = {0, 0};
  double least = 1e30;
  for (const Cost& c : costs) {
    const double rounds = mx8_row_blocks((double)rows / (double)n_slices, c.bm) * (double)(n_slices * ((N + c.bn - 1) / c.bn)) / 256.0;
    const double us = (ceil(rounds * 0.95) + ceil(rounds * 1.05)) * (c.start + (double)((K + 127) / 128) * c.stage);
    if (us < least) least = us, best = c.tile;
  }
  return best;
}

inline MxwTile mxw_tile(int64_t rows, int64_t n_slices, int64_t K, int64_t N, bool mx8) {
  const int64_t n256 = (N + 255) / 256, n512 = (N + 511) / 512;
  if (mx8) {
    if (rows > 104 * n_slices) return mx8_tile(rows, n_slices, K, N);
    if ((rows <= 96 * n_slices ? 256 * n_slices : 2 * rows + 128 * n_slices) * n256 <= 256 * 256) return {0, 0};  // (256ths of its row blocks)
    const int64_t alike = n_slices * n512;
    const bool few = alike < 3 * 256;
    if (few && rows <= 24 * n_slices) return {32, 256};
    return rows <= (alike > 192 && alike <= 256 ? 32 : 40) * n_slices ? MxwTile{64, 512} : MxwTile{128, 512};
  }
  if ((rows + 16 * n_slices) * n256 <= 512 * 32) return {32, 256};
  if (rows <= 20 * n_slices) return rows > 7 * n_slices && n_slices * n512 >= 3 * 256 ? MxwTile{64, 512} : MxwTile{32, 256};
  if ((rows + 160 * n_slices - 1) / (160 * n_slices) * n_slices * n512 < 512) return {64, 256};
  return rows <= 48 * n_slices ? MxwTile{64, 512} : rows <= 80 * n_slices ? MxwTile{96, 512} : MxwTile{160, 512};
}

// Whether 128 x 128 tiles of slices of 192 rows and more, half a row block a slice more than there are rows for, are one round of two workgroups a CU: they
// beat larger tiles, which then leave CUs without one or are little more than a round.  Measured (us, this kernel's 128 x 128 / the best of 256 x 256 and those of 320
// rows; slices, rows of one, K, N: 128 x 128 tiles).  bf16: 8, 272, 2048, 2048: 336 31.8 / 37.2; 8, 300: 364 33.5 / 38.1; 8, 400: 464 36.7 / 40.2; 8, 450, 1536: 514 32.6 / 34.2; 16, 272,
// 1024, 1280: 420 22.6 / 24.9; 16, 200, 1024, 1600: 429 26.1 / 25.6; 16, 400, 704, 896: 406 18.8 / 20.7 (256 x 256 30.7); 16, 300, 512, 1600: 591 31.6 / 29.1; 32, 200, 384, 1024: 528 18.5 /
// 18.0.  e4m3: 8, 272, 1536, 2048: 336 17.6 / 25.4; 8, 400, 2048, 2048: 464 23.0 / 30.6; 16, 272, 1024, 1152: 378 16.2 / 32.7; 16, 200, 6144, 1792: 462 64 / 68; 8, 272, 2048, 3072: 504
// 31.2 / 30.6; 8, 600, 1280, 2048: 664 26.8 / 25.9; 8, 272, 1024, 4096: 672 29.2 / 23.2; 16, 200, 1024, 2048: 528 17.8 / 21.7.
inline bool small_tiles_one_round(int64_t rows, int64_t n_slices, int64_t N) {
  return rows >= 192 * n_slices && (rows + 64 * n_slices) * ((N + 127) / 128) <= 500 * 128;
}

// Tile of the memory-to-LDS kernel (moe_gemm_dma_kernel.h) for 16-bit operands beside 256 x 256 ones: 320 rows, so that a slice of about 256 rows, of which
// a random routing makes half a few longer, is one row block.  (An eighth above the mean is 2.5 deviations at 400 rows, 2 at 256.)  rows 0 = those.
//   320 x 128 where its tiles are one round and 128 x 128 ones (above; up to 96 of 256 x 256, dma_block_n) are not better; 320 x 256 beyond, from 248 rows on.
// Measured (us of a GEMM with a random routing, 256 x 256 / 320 x 256 / 320 x 128; slices, K, N):
//   16, 2048, 4096: 224 rows 89 / 100 / 92, 240 101 / 95 / 92, 256 105 / 96 / 92, 272 130 / 101 / 107, 288 136 / 122 / 126, 320 142 / 150 / 152
//   16, 2048, 2048: 224 rows 56 / 72 / 50, 256 56 / 74 / 53, 272 57 / 78 / 58, 288 56 / 78 / 67; K 1024: 224 30 / 35 / 25, 272 32 / 40 / 28, 288 33 / 40 / 35
//   16, 2880, 2880: 240 rows 89 / 101 / 108, 256 111 / 102 / 111, 272 127 / 107 / 128; 32, 2048, 4096: 240 175 / 182 / 176, 256 225 / 184 / 181, 288 280 /
//   229 / 232; 32, 1024, 2048: 224 48 / 50 / 55, 256 65 / 55 / 59; 8, 4096, 4096: 224 102 / 120 / 83, 256 101 / 124 / 84, 272 103 / 132 / 108
//   8, 2048, 2048 (128 x 128 / 320 x 128): 256 30 / 34; 272 (256 x 256) 43 / 35; two blocks: 448 45 / 41, 544 47 / 43, 608 49 / 55
// (Slices that all have 256 rows to the row, or with favourites any number, are faster in the tiles of 256.  How a routing divides the rows is not known
// here: the kernel counts both kinds of tiles and goes on with the better one, moe_gemm_dma_tall.hip.)
struct DmaTile {
  int32_t rows, cols;
};
inline DmaTile dma_tile(int64_t rows, int64_t n_slices, int64_t N) {
  if (n_slices < 8 || small_tiles_one_round(rows, n_slices, N)) return {0, 0};
  const int64_t per_slice = rows / n_slices, n256 = (N + 255) / 256, blocks = (per_slice * 9 / 8 + 319) / 320;
  if (per_slice >= (blocks == 1 ? 192 : 448) && blocks <= 2 && n_slices * blocks * ((N + 127) / 128) <= 256 && n_slices * ((per_slice + 255) / 256) * n256 > 96)
    return {320, 128};
  return per_slice >= 248 && per_slice <= 288 && n_slices * n256 > 128 ? DmaTile{320, 256} : DmaTile{0, 0};
}

// Row blocks (of 64) that the kernel for few rows launches side by side: one a slice at least, and what slices of up to five quarters of
// the mean make, as a random routing does (at 62 rows per slice half of the slices have a second block).
inline int64_t few_row_blocks(int64_t rows, int64_t n_slices) { return n_slices * (rows * 5 / (n_slices * 256) + 1); }

// The decode layer row by row in two launches (moe_decode_rows.hip; up to kDecRowsMaxK experts a token), which keep nothing between calls: where that
// is the smaller stream.  The single launch costs some 30 us around its stream but reads an expert once; the two launches cost 4, but they read
// an expert's weights (padded, as they lie in memory) again for each of its rows, at about 4 MB/us, and the second one's workgroups, one for a token and
// 16 columns, take 5.5 ns each, as long as 22 KB do.  The more rows, the more of them share an expert, which nobody knows here: 1 MB a row.
// Measured (us, row by row against single launch, with all experts alike; with a few that most tokens choose), at MB of this sum:
//   d and d_ff 2880, 128 experts: 8 rows, top 4, 124 MB, 31 / 38; 30 / 37; 10 rows, top 2, 165, 38 / 42; 33 / 39; 12, top 4, 186, 44 / 45; 40 / 40
//   2048, 64 experts: 16, top 1, 168, 36 / 41; 33 / 34; 20, top 2, 182, 36 / 45; 32 / 36; 21, top 1, 221, 46 / 46; 41 / 35; 26, top 2, 236, 46 / 50; 40 / 38
//   1536, 32 experts: 32, top 8, 161, 36 / 44; 35 / 38; 24, top 1, 165, 35 / 39; 31 / 32; 40, top 2, 233, 37 / 42; 35 / 31; 32, top 1, 220, 44 / 42; 40 / 33
//   1024, 32 experts: 48, top 2, 162, 31 / 40; 28 / 31; 64, top 8, 182, 36 / 41; 35 / 36; 64, top 2, 216, 39 / 41; 35 / 31; 48, top 1, 196, 41 / 41; 36 / 32;
//     64, top 1, 261, 51 / 42; 47 / 32
//   1024 and 2048, 8 experts: 32, top 2, 162, 30 / 31; 29 / 31; 32, top 1, 184, 36 / 31; 33 / 30
//   512, 32 experts: 64, top 1, 136, 26 / 31; 26 / 29
// (A caller that names a spin limit asks for the launch whose waits it bounds.)
constexpr int kDecRowsMaxK = 8;
inline bool decode_by_rows(int64_t T, int64_t k, int64_t d_ff, int64_t d_model) {
  constexpr int64_t kRowsMax = 64, kRowsBytes = 183'000'000, kWorkgroupBytes = 22'000, kRowBytes = 1'000'000;
  auto parts = [](int64_t n, int64_t of) { return (n + of - 1) / of; };
  const int64_t expert_bytes = (parts(2 * d_ff, 32) * parts(d_model, 128) + parts(d_model, 32) * parts(d_ff, 128)) * (2048 + 128);
  return k <= kDecRowsMaxK && T * k <= kRowsMax && T * k * (expert_bytes + kRowBytes) + T * parts(d_model, 16) * kWorkgroupBytes <= kRowsBytes;
}

// How a decode layer in a single launch fetches the weights.  Up to 16 tokens no expert has a second row block (a token's k experts differ): they are read once by the whole grid,
// with the non-temporal hint, which is the faster way wherever other layers run in between (us, plain loads / with the hint, the same weights again and again; other weights
// each call: 16 tokens, 16 experts, top 4, 2048 36.3 / 36.2; 38.7 / 37.4; 16, 8, top 4, 2880 37.4 / 38.6; 40.4 / 39.8; 10, 8, top 8, 2880 39.8 / 40.8; 42.6 / 41.9; 16, 32, top 8, 1024 31.7 / 30.9; 32.5 / 32.1;
// 16, 64, top 8, 768 33.3 / 33.3; 34.1 / 33.5).  Beyond, the later row blocks of an expert find a fragment in the caches that the hint would take away: up to kLargeBlocks, plain loads; where there
// may be more than the caches keep for the next call anyway, the kernel decides, which knows the blocks after its routing: hardly any second ones, all with the hint; up to a third, by unit
// (whole K of 24 stages only: the branch costs the compiler's wait counts, a drained ring a unit, which shorter units feel more than they gain).  Three
// copies of the loop are code to be fetched (0.8 us a call for those behind the first), so the host rules out what cannot be.
// us, 128 experts, top 4, 2880, without and with: no second blocks, 17 tokens 143 / 130, 32 215 / 192, 64 291 / 260; with favourites, 32 tokens (27.6 blocks of
// 25.7 experts) 90.5 / 83.6, 40 (32.8 of 30.4) 96.5 / 93.0, by unit 89.5, 61 (39.9 of 33.9) 117.2 / 119.1, by unit 111.5; 33 tokens, 96 experts, 768 and 1824, favourites, 100 MB 37.9 / 40.5.
enum { kFetchPlain, kFetchOnce, kFetchEither };
constexpr int kLargeBlocks = (128 << 20) / 2176;  // blocks of 32 columns x 128 k, values and scales
inline int decode_fetch(int64_t T, int64_t k, int64_t E, int64_t blocks_of_expert) {
  if (T <= 16) return kFetchOnce;
  return (T * k < E ? T * k : E) * blocks_of_expert <= kLargeBlocks ? kFetchPlain : kFetchEither;
}

// Tile of the ragged-K kernel for long slices (ragged_k_long.hip) for aligned operands, `k` a slice; 0 = the one for short slices, whose four small workgroups a CU write best where
// writing is what takes the time.
//   * From 160 k a slice on 256 x 256 where they are four rounds over the 256 CUs; with fewer, 128 x 128, which start sooner.
//   * From 90 k on 256 x 256 or nothing: where they are 24 rounds (below: 16 slices of 128, 2880, 17 rounds for the larger product, lose; 32, 34 rounds, gain) and
//     an eighth of their area at most hangs over the edges (1600 x 2400, a fifth, loses).  2880 x 2880 and 1440 x 2880, 0.138, are beyond that line, so of the layers of 2880 with 90 to 160 k only the
//     product of 2880 x 5760 (0.094) is this kernel's, and neither of those of 1440: the table's columns are both products by one kernel (128 slices of 128, 2880: by this rule 1642).
// Measured (us of both products [d, 2 f] and [f, d] of a layer with slices of random lengths; short / 128 / 256):
//   slices, k of one, d, f: 8, 2048, 2880, 2880 936 / 916 / 827; 8, 256, 2880, 2880 162 / 163 / 155; 16, 1024, 2048, 2048 498 / 491 / 423; 16, 375, 1600, 1200 121 / 110 / 110
//   32, 512, 2880, 2880 1069 / 1104 / 935; 32, 187, 2880, 2880 477 / 512 / 464; 32, 187, 1600, 1200 135 / 132 / 135; 64, 256, 1024, 1024 168 / 172 / 146; 64, 256, 2880, 2880 1309 / 1357 / 1149
//   8, 2048, 512, 512 132 / 85 / 192; 8, 256, 512, 512 26 / 21 / 40; 8, 2048, 1024, 1024 162 / 134 / 210; 8, 750, 800, 1024 71 / 55 / 87; 16, 375, 320, 448 39 / 30 / 54; 16, 256,
//   1024, 1024 60 / 47 / 55; 32, 187, 320, 448 35 / 30 / 48; 32, 187, 800, 1024 77 / 69 / 73; 64, 256, 320, 448 50 / 47 / 54
//   128, 128, 2880, 2880 1742 / 1903 / 1623; 128, 128, 1440, 1440 456 / 472 / 421; 64, 93, 2880, 2880 706 / 733 / 681; 32, 128, 2880, 2880 407 / 418 / 396; 16, 128, 2880, 2880 202 / 223 / 208
//   128, 128, 1600, 1200 404 / 438 / 411; 64, 93, 1600, 1200 184 / 196 / 197; 64, 125, 1440, 1440 226 / 242 / 231; 8, 128, 512, 512 15 / 14 / 23; 128, 128, 512, 512 76 / 82 / 76; 128, 46, 2880,
//   2880 1171 / 1275 / 1221; 16, 64, 1600, 1200 25 / 29 / 30
constexpr int kRaggedKLongSlices = 128;  // slices that the kernel for long ones keeps in registers
inline int ragged_k_tile(int64_t k, int64_t M, int64_t N, int64_t n_slices) {
  if (n_slices > kRaggedKLongSlices) return 0;
  const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256) * n_slices;
  if (k >= 160) return tiles >= 4 * 256 ? 256 : 128;
  return k >= 90 && tiles >= 24 * 256 && tiles * 256 * 256 * 8 <= M * N * n_slices * 9 ? 256 : 0;
}

}  // namespace tk
