// Rules by which a default variant chooses a kernel or a launch shape from the sizes of a call: plain functions of whole numbers, free of HIP
// calls, so that a test can evaluate them on a host.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define DISPATCH_FN __host__ __device__ __forceinline__
#else
#define DISPATCH_FN inline
#endif

namespace dispatch {

// ---- GEMM: the order in which the workgroups take the tiles ----
// Workgroup -> tile.  Workgroup b runs on XCD b % 8.  `walk` is what tile_walk() chose: blocks, row-major, or the rows of a band.
constexpr int kWalkBlocks = 0, kWalkRowMajor = -1;
DISPATCH_FN void tile_of_workgroup(const int b, const int tiles_m, const int tiles_n, const int walk, int& tile_m, int& tile_n)
{
  const int xcd = b & 7, idx = b >> 3;
  if (walk == kWalkBlocks) {
    const int bm = tiles_m / 4, bn = tiles_n / 2;       // block of one XCD
    tile_m = (xcd >> 1) * bm + idx / bn;
    tile_n = (xcd & 1) * bn + idx % bn;
  } else if (walk == kWalkRowMajor) {
    tile_m = b / tiles_n;
    tile_n = b % tiles_n;
  } else {
    const int rows = walk, tiles = tiles_m * tiles_n, each = tiles >> 3, more = tiles & 7;
    const int at = xcd * each + (xcd < more ? xcd : more) + idx;
    const int band = at / (rows * tiles_n), in_band = at - band * rows * tiles_n;
    const int height = tiles_m - band * rows < rows ? tiles_m - band * rows : rows;
    tile_n = in_band / height;
    tile_m = band * rows + in_band - tile_n * height;
  }
}

// `per_cu` workgroups share one of `cus` compute units.  Every XCD has an L2 of its own, so the panels of A and B behind the tiles that are in
// work on one XCD at a time should be few.
//   blocks     grids that divide into 4 x 2: every XCD gets one compact block, unless the grid is narrow (below).
//   bands      up to eight tile rows, down the columns of a band, an eighth of that walk for every XCD (dealt row-major instead:
//              3712 x 4736 x 3712 with 128 x 128 tiles 188 us against 139, 640 x 8064 x 2048 34 / 28).  In grids that divide level or slower than
//              blocks (8192 x 8192 x 1024, 256 x 256 tiles: 155 us against 140).
//   row-major  where eight divides the tiles of a row, so that every XCD has columns of its own, and its rows and columns are then no more
//              than with bands (7680 x 8192 x 384, 256 x 256 tiles: 79 us, bands 87; 640 x 8192 x 1024, 128 x 128: 15.5 / 16.8.  But
//              16 rows and 4 columns against 8 and 8: 3712 x 4096 x 640 33.5 / 28.8 from DRAM; 15 and 2 against 6 and 5: 1920 x 2048 x 2048
//              26.6 / 23.0.  Tiles below 128 x 128 compare with the rows that the grid has, two or four often, in bands of which B is what counts: bands /
//              row-major 256 x 5120 x 2432 24 % and 31 %, 256 x 7680 x 512 3 % and 21 %, 128 x 9728 x 512 3 % and 25 %; with 128 x 128 the same count would
//              lose, 640 x 11264 x 7040 6 % and 8 %); where one round of tiles is over in a few K steps and finding the place in a band counts (0.2 us: 640 x 4096 x 256
//              5.4 / 5.6); and with two K steps of 64, when a tile is mostly its block of C and the bands scatter the writes of a large C, as long as
//              an L2 holds B (from DRAM: 8064 x 8064 x 128 49 / 55, 4224 x 5760 x 128 20.7 / 22.9; 6528 x 896 x 128, a small C, 8.0 / 7.5;
//              2176 x 7808 x 256 24.4 / 21.9).
// Narrow grids: the blocks of a grid of few tile rows are strips that touch many more panels than a band's share.  What such a grid walks in
// instead depends on what it would walk in if it did not divide.  us, from the caches and from DRAM, blocks / that walk, tiles of 128 x 128:
//   own columns    from 13/7 times the panels (1024 x 6144 x 2048 31.7 / 28.1 and 41.4 / 35.1, 512 x 8192 x 4096 42.9 / 35.1 and 46.1 / 42.9; but 1.83
//                  times, 1024 x 5120 x 1024, 17.9 / 16.8 and 18.1 / 20.4), or from 1.5 and k = 2048 on if the bands' last one would be no thin
//                  rest (1536 x 8192 x 2048 19 % and 9 %, 2048 x 10240 x 2048 104 / 85 and 111 / 99).  Among grids of ten columns an XCD 1024 x 10240 x 512
//                  still loses from DRAM (9 %; 13 % faster from the caches).
//   bands of four  the whole height: from 1.8 times (512 x 16384 x 512 17.8 / 12.3 and 21.3 / 17.9, 512 x 8448 x 2048 22 % and 44 %).
//   one band of    eight: from 2.5 times and k = 1024 on (1024 x 11776 x 2048 14 % and 2 %); below, the caches gain a tenth and DRAM loses
//                  up to 18 % (1024 x 6912 x 512 1 % and -18 %, x 4096 7 % and -5 %).  Of seven and a thin rest: never (1024 x 5632 x 512 10.2 / 11.6 and
//                  14.5 / 16.1).
//   more bands     from 13/7 times and k = 1024 on (1536 x 11008 x 1536 15 % and 9 %; 1536 x 9984 x 512 15 % and -8 %), or from 1.5 times and k = 2048 on if
//                  they divide the rows evenly (2048 x 8960 x 2048 91 / 79 and 101 / 95; with half a band left over 1536 x 7424 x 2048 6 % and -9 %).
// Tiles below 128 x 128 are taken for products that are over soon: from 1.8 times at every k (128 x 4096 x 1024 6.0 / 5.0 and 9.1 / 7.7), and from 1.5
// times and k = 2048 on without a thin rest (5376 x 256 x 2048 15.6 / 14.3 and 19.5 / 17.3).
inline int tile_walk(const int m, const int n, const int k, const int tile_rows, const int tile_cols, const int per_cu, const int cus)
{
  const int tiles_m = m / tile_rows, tiles_n = n / tile_cols;
  const long long tiles = (long long)tiles_m * tiles_n, each = tiles / 8;
  int rows = 1;
  while (rows < 8 && rows * rows < each) ++rows;
  const double in_work = (double)(each < per_cu * cus / 8 ? each : per_cu * cus / 8), columns = tiles_n / 8;
  const int high = tiles_m < rows ? tiles_m : rows, rest = tiles_m % rows, height = tile_rows < 128 ? high : rows;
  const bool own_columns = (tiles_n % 8) == 0 && in_work / columns + columns <= height + in_work / height + 1;
  const bool mostly_c = k < 256 && (long long)n * k < (3 << 19) && (long long)m * n >= (16 << 20);
  const int other = own_columns || mostly_c || (tiles <= cus && k < 512) ? kWalkRowMajor : rows;
  if ((tiles_m % 4) != 0 || (tiles_n % 2) != 0) return other;

  const long long of_block = tiles_m / 4 + tiles_n / 2, of_band = high + each / high;        // panels behind a block and behind a band's share
  const bool times_1_5 = 2 * of_block > 3 * of_band, times_1_8 = 5 * of_block > 9 * of_band, times_13_7 = 7 * of_block >= 13 * of_band,
             times_2_5 = 2 * of_block >= 5 * of_band;
  const bool thin_rest = rest != 0 && 2 * rest < rows;
  bool narrow;
  if (tile_rows < 128) narrow = times_1_8 || (times_1_5 && k >= 2048 && !thin_rest);
  else if (tiles_m == 4) narrow = times_1_8 && k >= 512;
  else if (other == kWalkRowMajor) narrow = (times_13_7 && k >= 512) || (times_1_5 && k >= 2048 && !thin_rest);
  else if (tiles_m == 8) narrow = times_2_5 && k >= 1024 && rest == 0;
  else narrow = (times_13_7 && k >= 1024) || (times_1_5 && k >= 2048 && rest == 0);
  return narrow ? other : kWalkBlocks;
}

// ---- GEMM: the kernel of the default variant ----
// Whether the rows of one round of direct-to-LDS loads (32 of A, 16 of B) span less than the 4 GiB of a lane offset.
inline bool direct_rows_fit(const long long n, const long long k)
{
  return 32 * (k * 2) + 128 <= 0xffffffffLL && 16 * (n * 2) + 256 <= 0xffffffffLL;
}

enum class GemmForm { kLongRows, kDealt32x32, kDealt32x64, kDealt64x64, kDealt64x64Two, k128Far, k128, k256 };
inline GemmForm gemm_form(const int m, const int n, const int k, const int compute_units)
{
  const long long cus = compute_units;
  // Longer rows go through variant 1, whose transfers take a 64-bit offset for every row.
  if (!direct_rows_fit(n, k)) return GemmForm::kLongRows;

  // Grids of few tiles take the smallest tile that still gives every compute unit at most one (32 x 32, 32 x 64, 64 x 64) or, with half as
  // many wavefronts, two workgroups (64 x 64).  us with those four and with 128 x 128, from the caches: 512 x 512 x 512 3.5 / 3.7 / 4.6 / 4.6 / 6.0;
  // 640 x 512 x 1152 6.0 / 4.8 / 6.0 / 6.4 / 9.8; 768^3 6.7 / 7.0 / 5.3 / 5.5 / 7.8; 1024 x 1152 x 1920 - / - / 15.2 / 12.6 / 14.8 and from DRAM
  // 17.0 / 14.8 / 20.4.  The last one has a wavefront only two or three steps below k = 512, and
  // then 128 x 128 is as fast or faster (1152 x 1792 x 256 from the caches 5.5 / 5.1, from DRAM 5.9 / 5.7; x 512 6.4 / 6.6 and 7.0 / 7.5; x 768 7.7 / 8.1 and 8.8 / 10.0).
  // With long rows 128 x 128 has caught up (256 x 6656 x 6144 45.0 / 42.0 and 63.4 / 61.3; 768 x 2560 x 3072 24.0 / 22.3 and 29.7 / 30.7); where
  // nearly every compute unit has two of them it does so from k = 1900 on from the caches, not from DRAM (1152 x 1536 x 2304 18.8 / 17.4 and 19.7 / 23.8,
  // 768 x 2432 x 1920 15.7 / 15.2 and 18.5 / 20.5, 3968 x 512 x 2176 16.9 / 16.8 and 19.6 / 23.3).  A product of two rows of more than 80 of them is nearly all B, which a tile of 64 columns fetches in pieces of
  // 128 bytes: 128 x 128 is ahead there from k = 1024 on (128 x 11776 x 2176 10 % and 8 %, 128 x 14464 x 1664 5 % and 4 %, 128 x 16384 x 1024 0 % and 7 %; 128 x 10624 x 1536
  // 2 % slower and 1 % faster.  With 80 128 x 10240 x 1792 is 7 % and 19 % slower).
  const long long t32 = (long long)(m / 32) * (n / 32);
  if (t32 <= cus) return GemmForm::kDealt32x32;
  if (t32 <= 2 * cus) return GemmForm::kDealt32x64;
  if (t32 <= 4 * cus) return GemmForm::kDealt64x64;
  if (t32 <= 8 * cus && k >= 512 && k < (m == 128 && t32 > 5 * cus ? 1024 : 3072)) return GemmForm::kDealt64x64Two;

  // Variant 9 with its tile of 256 x 256 or the same kernel with 128 x 128, whichever takes its rounds over the compute units in less time.
  // `full` is the time of a K step of 64 of a whole round in units of 10 ns, `part` that of a round of few workgroups: up to one per
  // compute unit for the small tile, of which two share one, up to five eighths of them for the large one (they get more of the
  // clock and the memory); `once` is what a tile costs before its first and after its last K step.  Measured, 256 / 128:
  // 1536 x 7680 x 1280 38 / 44 us, 2816 x 5888 x 1024 39 / 42, 7424 x 2304 x 2048 99 / 81, 2048^3 41 / 23, 2560 x 2560 x 1024 25 / 18.  The tiles of variants 2 and 3
  // lie between and win nowhere.
  auto rounds = [&](const long long tiles, const long long slots, const long long few, const int full, const int part, const int once) {
    const long long rest = tiles % slots;
    return (k / 64) * (tiles / slots * full + (rest == 0 ? 0 : rest <= few ? part : full)) + once;
  };
  const long long grid = (long long)(m / 128) * (n / 128);
  const long long small = rounds(grid, 2 * cus, cus, 100, 58, 400);
  const bool even = (m % 256) == 0 && (n % 256) == 0;
  if (even && rounds((long long)(m / 256) * (n / 256), cus, cus * 5 / 8, 160, 110, 1000) < small) return GemmForm::k256;
  // One tile or none for a compute unit: requests that run further ahead, from the k on at which <2, 4> loses from DRAM what it gained
  // over the warp-specialised kernel (us, <2, 4> / <2, 8> from the caches, <2, 4> / <2, 8> / variant 1 from DRAM): 2048 x 2048 x 640
  // 9.4 / 9.9, 10.2 / 10.3 / 10.6; x 768 10.3 / 10.5, 13.4 / 12.3 / 12.3; x 1280 15.1 / 15.2, 19.2 / 17.1 / 16.9; x 2048 23.3 / 20.9,
  // 28.7 / 24.2 / 24.6; 768 x 2048 x 4736 40 / 33, 56 / 45.
  return grid <= cus && k >= 768 ? GemmForm::k128Far : GemmForm::k128;
}

// ---- copy: the kernel of the default variant ----
// Two operating points, as for every read + write stream on this part: a working set (both buffers) that the 256 MB Infinity
// Cache holds from launch to launch wants many tiles in flight (two LDS tiles, four workgroups per compute unit);
// beyond it the memory system serves a short queue better (one LDS tile, two workgroups per compute unit: 1 GiB in 0.353 ms
// against 0.408 ms).  Stores are non-temporal throughout, which leaves the caches to the input.  us from the caches, from DRAM, and with three sets of
// buffers in turn, of which the caches hold a part:
//            plain stores, two tiles    one tile, four workgroups    two tiles, streaming loads    two tiles, plain loads
//   16 MiB   5.6   7.5   7.3            5.5   6.1   5.6              5.5   6.3   5.7               4.4   6.4   6.8
//   32 MiB   11.2  11.7  10.9           11.2  12.5  12.0             9.6   11.9  11.4              8.9   11.6  11.5
//   40 MiB   13.3  18.2  13.2           13.3  15.3  14.8             13.0  14.8  14.2              13.9  15.4  13.6
//   44 MiB   14.5  18.4  16.5           14.7  16.6  16.0             14.4 to 15.6  16.0  15.4      15.0  16.8  14.7
//   46 MiB   15.3  20.7  18.0           15.3  17.3  16.6             15.2 to 16.9  17.5  16.8      15.7  18.2  15.4
//   48 MiB   15.8  21.3  20.5           16.6  17.9  17.4             15.8 to 17.5  17.7  17.2      16.2  18.3  15.9
//   64 MiB   20.9  25.0  24.8           22.1  23.4  22.7             21.1 to 23.6  24.1  23.3      21.1  24.8  20.7
//   96 MiB   30.6  39.0  38.3           32.2  34.0  33.2             32.5  34.4  33.0              30.7  35.9  33.9
// Up to 16 MiB the one tile starts sooner with inputs that come from memory.  Streaming loads end at 44 MiB: beyond, they lose up to a tenth
// with the same buffer again and again, by where it lies, and as much with three in turn.
constexpr unsigned long long kCacheAssistedBytes = 192ull << 20;
enum class CopyForm { kOneTileFour, kTwoTilesStreaming, kTwoTiles, kOneTileTwo };
inline CopyForm copy_form(const unsigned long long bytes)
{
  if (bytes <= 16ull << 20) return CopyForm::kOneTileFour;
  if (bytes <= 44ull << 20) return CopyForm::kTwoTilesStreaming;
  return 2 * bytes <= kCacheAssistedBytes ? CopyForm::kTwoTiles : CopyForm::kOneTileTwo;
}

// ---- row sums of a gather, four tiles in a transfer: workgroups per compute unit ----
// Four where the Infinity Cache holds the table or the call is over soon.  A larger table wants a shorter queue; how short is a matter of a few
// per cent (us with two / three / four, from the caches where they hold a part):
//   384 MiB  2 Mi indices 44.3 / 44.6 / 44.7   8 Mi 162.8 / 166.8 / 168.3   32 Mi 628 / 645 / 653
//   640 MiB  2 Mi 46.1 / 44.9 / 45.2           8 Mi 159.7 / 163.4 / 165.1   32 Mi 618 / 627 / 636
//   768 MiB  4 Mi 84.6 / 88.6 / 88.7           8 Mi 163.2 / 161.5 / 162.1   32 Mi 637 / 627 / 636
//   1 GiB    4 Mi 86.0 / 86.6 / 87.1           8 Mi 173.7 / 165.9 / 167.2   16 Mi 335 / 324 / 328
//   1.5 GiB  8 Mi 182.1 / 176.0 / 177.3        4 GiB  2 Mi 45.6 / 46.4 / 47.4 (from DRAM 54.6 / 52.4 / 52.7)   16 Mi 392 / 384 / 390
// From DRAM three are level or ahead by up to 5 % below 4 Mi indices and behind by 3 % beyond 8 Mi up to 512 MiB.
inline int rowsum_workgroups(const unsigned long long table_bytes, const unsigned long long n_idx)
{
  if (table_bytes <= 256ull << 20 || n_idx <= 1ull << 20) return 4;
  return table_bytes <= 640ull << 20 || (table_bytes <= 1ull << 30 && n_idx <= 6ull << 20) ? 2 : 3;
}

}  // namespace dispatch
