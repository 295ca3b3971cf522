// Which tiles or kernel the casts down the columns take, and the order in which the one-read casts go over their tiles: plain arithmetic on
// sizes, without the device.
#pragma once

#include <stdint.h>

#include "dt_host.hpp"

namespace dt {

constexpr int kDualRows = 128;

// MXFP8 down the columns (mx_dual_kernel without its row-wise half): tiles of 128 rows x 128 columns (fp32: 64), or twice as wide.
// Narrow tiles fill the chip where tiles are few, and the 16-bit ones also beat the walking grid where there are many (us, wide ->
// narrow, bf16: 512 x 512 4.4 -> 3.4, 1024 x 1664 5.3 -> 4.3, 2048 x 1888 6.3 -> 5.5, 2752 x 4096, 352 tiles, 9.3 -> 8.8, 3584 x 8192, 896
// tiles, 18.9 -> 17.8, 8192 x 8192 40.8 -> 38.1, 4096 x 14336 35.2 -> 32.4; fp32: 512 x 512 3.4 -> 3.0, 2048 x 4096, 512 tiles, 9.8 -> 9.3).
// In between, and for more fp32 tiles, the wide ones win (bf16 4096 x 3488, 448 tiles, 10.6 and 11.3, 6144 x 4096, 768 tiles, 15.5 and
// 16.4; fp32 4096 x 4096 17.1 and 18.1, 8192 x 8192 58.9 and 61.6).
// Row-major scales: the many narrow ones lose where a column's scale bytes are no whole words (6240 x 11968 50.3 and 53.7) and in matrices
// four times as tall as wide (16384 x 4096 39.3 and 39.9; 14336 x 4096 35.9 -> 34.5).
// fp32, blocked scales: of up to 64 columns every other narrow tile holds nothing but the padding of the scales to 128 columns, which
// loses once they are more than one per CU (8192 x 64 4.1 -> 3.8, 16384 x 64 4.3 and 4.3, 20480 x 64 4.5 and 5.0, 65536 x 64 6.6 and 8.1; three
// tiles of four, 20480 x 192 7.2 -> 6.8).
inline bool narrow_cols(bool f32, bool blocked, int64_t rows, int64_t cols, int64_t cus) {
  const int64_t tiles = ceil_div(rows, (int64_t)kDualRows) * ceil_div(cols, (int64_t)(f32 ? 128 : 256));  // wide ones
  if (f32) return tiles <= (blocked && cols <= 64 ? cus / 2 : 2 * cus);
  return tiles * 8 <= 11 * cus || (tiles * 2 >= 7 * cus && (blocked || (rows % 128 == 0 && rows < 4 * cols)));
}

// mx_col_t_kernel; or mx_dual_kernel without its row-wise half, on tiles of 128 rows x 256 columns by a grid of walking workgroups, where 16-bit
// tiles are more than that grid (us, it / mx_col_t_kernel, bf16: 8192 x 8192 33.1 / 33.9, 16384 x 4096 30.5 / 35.5; fp32 55.4 / 51.9); or the same on
// tiles half as wide (256 -> 128 columns, fp32 128 -> 64), one workgroup each:
//  - where tiles are few, the narrow ones fill the chip (us, before -> narrow, bf16 512 x 512 3.9 -> 3.2, 1024 x 1664 4.5 -> 4.1; not of 32 rows, 32 x
//    15840 3.4 and 3.7, nor 2432 x 3104, 247 tiles, 6.1 and 7.0; fp32 512 x 512 4.7 -> 3.1, 2048 x 2048 6.5 -> 5.9; not 2560 x 3072, 480 tiles, 7.9 and 8.7);
//  - fp32, just past two tiles per CU, where the others begin another round (2560 x 3584, 560 tiles, 11.5 -> 9.6), and where there are more and the
//    transposed rows are off the cache lines (12320 x 2368 30.0 -> 26.7, 7328 x 8288 69.3 -> 56.5; 8192 x 8192 54.6 and 60.0);
//  - 16 bits, more than one and up to one and a half per CU, of a matrix that is not four times as tall as wide (3104 x 3264 9.4 -> 7.9, 672 x 14304
//    9.9 -> 8.3; 14592 x 672 8.0 and 8.2), and more than four per CU of one sixteen times as tall (54944 x 736 29.3 -> 24.7, 85792 x 864 48.9 -> 43.6);
//  - 16 bits, more than one per CU, where the rows of x begin on lines (6240 x 11968 38.1 -> 36.5, 3072 x 4096 9.0 -> 7.9; 12320 x 4064 31.4 and 36.3,
//    4960 x 16416 51.3 and 60.4), the transposed payload goes out in whole pieces of 64 bytes (row-major scales 16608 x 704 10.0 and 13.5,
//    5056 x 21056 60.8 and 66.6), and the walking grid, if it is one, does not go in bands of row tiles (12288 x 6144 38.1 and 43.2).
// Picked from all three at 751 sizes of 0.25 to 130 million elements, half of them round, bf16 and fp32, both layouts of the scales: 0.95 / 0.91
// (bf16 / fp32) of the time that the first two alone take, at no size more than 1.1; at 126 others, 0.92 and 1.08.
// pipe_grid: workgroups of the walking grid; forced: the knob mx.dual_narrow.
enum Fp4Cols { kFp4ColT, kFp4Wide, kFp4Narrow };
inline Fp4Cols plan_fp4_cols(bool f32, bool blocked, int64_t rows, int64_t cols, int64_t cus, int64_t pipe_grid, int forced) {
  const int64_t tiles = ceil_div(rows, (int64_t)kDualRows) * ceil_div(cols, (int64_t)(f32 ? 128 : 256));
  bool narrow;
  if (forced >= 0)
    narrow = forced != 0;
  else if (f32)
    narrow = tiles <= cus || (tiles > 2 * cus && (2 * tiles <= 5 * cus || rows % 128 != 0));
  else
    narrow = (2 * tiles <= cus && rows > 32) || (tiles > cus && 2 * tiles <= 3 * cus && rows < 4 * cols) ||
             (tiles > 4 * cus && rows > 16 * cols) ||
             (tiles > cus && cols % 64 == 0 && (rows % 128 == 0 || (blocked && tiles > 4 * cus)) &&
              (tiles <= 2 * cus || rows % (8 * kDualRows) != 0));
  return narrow ? kFp4Narrow : !f32 && pipe_grid > 0 && tiles > pipe_grid ? kFp4Wide : kFp4ColT;
}

// Tile order of the casts along both axes from one read: 0 = down the rows first, 1 = along the columns first, 2 = bands of 8 row tiles.  Along the
// columns first (us, against down the rows: bf16 wide tiles 16384 x 4096 51.6 and 58.7, narrow ones 48.5 and 58.6, fp32 3840 x 10784 50.7 and 66.9);
// down the rows first for matrices four times as wide as tall (narrow tiles, 2976 x 11968 30.8 and 32.0), and for fp32 ones of rows that
// lie multiples of 32 KiB apart already from twice, while the tiles are not many (3584 x 8192 MXFP8 36.1 against 37.3, MXFP4 31.5 against 33.6; 5120
// x 16384, 5120 tiles, 94.4 and 87.4); wide tiles of MXFP4 in bands where the row count allows and there are three per CU or more (against along
// the columns, bf16 16384 x 2560 28.3 and 30.2, fp32 8192 x 2560 22.9 and 24.0; 14336 x 1024, 448 tiles, 12.0 and 11.4).
inline int pair_order(bool f32, bool fp4, bool narrow, int64_t rows, int64_t cols, int64_t cus) {
  const int64_t tiles = ceil_div(rows, (int64_t)kDualRows) * ceil_div(cols, (int64_t)(f32 ? 128 : 256));  // wide ones
  if (cols > 4 * rows || (f32 && cols > 2 * rows && cols % 8192 == 0 && tiles <= 8 * cus)) return 0;
  return fp4 && !narrow && rows % (8 * kDualRows) == 0 && cols <= 2 * rows && tiles >= 3 * cus ? 2 : 1;
}

}  // namespace dt
