// Which kernel and tiles a block-scaled product runs on, and how many workgroups share a tile's K: plain arithmetic on sizes, without the
// device.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "dt_host.hpp"
#include "mx_few_lines.hpp"

namespace dt {

constexpr int kBK = 128;             // K bytes per step = one 16x16x128 MFMA
constexpr size_t kSplitTicketBytes = 1024;        // head of the split-K workspace: one counter per tile, 256 at most
constexpr size_t kSplitTileBytes = 128 * 128 * 4;  // the rest: parked fp32 accumulators, room for one 128 x 128 tile per CU
constexpr int kMaxSplits = 16;      // what gemm.split_k may force
constexpr int kAutoMaxSplits = 12;  // what the library picks by itself

enum GemmTiles {
  kSmallTiles,               // the kernel for few tiles, in the form that plan_ring gives
  kTiles256Halves,           // 256 x 128 halves of 256 x 256 tiles
  kTiles256x192,
  kTiles256,
  kTiles256ThenQuads,        // whole rounds of 256 x 256, the tiles left over as 128 x 128 quadrants
  kTiles256ThenHalves,       // or as halves
  kTiles256QuadrantSchedule,  // 256 x 256 on the other tiles' main loop (on request only)
  kFewRows,                  // the kernel for at most 64 rows that loads B into registers (mx_few_rows.hip)
  kFewLines                  // the one for at most 32 rows by whole lines, in the form that plan_few_lines gives
};

// The tiles of a product by its size, without the kernel for few rows.  variant, tail: the knobs gemm.variant and gemm.tail_quads.
inline GemmTiles plan_tiles(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, int cus, int variant, int tail) {
  const int64_t tiles256 = ceil_div(M, 256) * ceil_div(N, 256);
  // 256 x 192 tiles where they fill the chip's one round better than 256 x 256 tiles do (which leave a
  // quarter of it idle or more).  At the chip's power limit a round of them takes 0.78 of a round of the
  // large tiles, not 0.75, so they only pay while both are one round (us, 256 x 256 -> 256 x 192, e4m3 and
  // e2m1: 2048 x 4352 x 4096, 136 -> 184 tiles, 38.5 -> 34.3 and 26.0 -> 23.6; 2048 x 5120 x 5120, 160 -> 216,
  // 48.3 -> 45.3 and 30.9 -> 29.3; 2000 x 6144 x 8192, 192 -> 256, 80.0 -> 77.7 and 50.9 -> 49.2; two rounds
  // against one and a half: 4096 x 5632 x 4096 77.9 and 77.9, 4096 x 9216 x 4096 120.9 -> 123.5).
  const int64_t tiles192 = ceil_div(M, 256) * ceil_div(N, 192);
  if (variant == 5 || (variant == 0 && 2 * tiles256 > cus && tiles192 > tiles256 && tiles192 <= cus)) return kTiles256x192;
  if (variant == 2) return kTiles256;
  if (variant == 7) return kTiles256QuadrantSchedule;
  // One round of 128 x 128 tiles is taken before anything larger.  Between a quarter and half a round of
  // 256 x 256 tiles: as 256 x 128 halves they fill the chip once (0.8 of a round of tiles), as 128 x 128 tiles
  // two rounds (2 x 0.55) unless rows or columns past the matrix leave much of the large tiles idle.  With at
  // most 128 rows (or an odd number of 128-row bands) that may be one round, which is the shorter one then, also
  // at exactly half a round of the large tiles (us, halves -> 128 x 128, e4m3 and e2m1: 96 x 28672 x 4096
  // 34.6 -> 30.6 and 21.4 -> 16.9, 128 x 32768 x 4096 39.5 -> 35.7 and 24.9 -> 19.3 where 256 x 256 tiles take 53.1
  // and 32.3, 1152 x 3584 x 4096 26.4 -> 22.7 and 19.3 -> 15.9).
  if (variant == 0 && ceil_div(M, 128) * ceil_div(N, 128) > cus) {
    // Rows off the cache lines cost the halves two requests a line, the small tiles one more window (us, halves -> 128 x 128, operands from
    // the memory-side cache / from memory: e4m3 520 x 10704 x 2016 24.1 -> 21.1 / 28.4 -> 25.7, 986 x 4808 x 2464 26.5 -> 24.2 / 31.9 -> 26.3,
    // 726 x 9072 x 9952 105.8 -> 93.1 / 106.2 -> 94.8; e2m1 1292 x 5232 x 10304 55.7 -> 51.2 / 67.6 -> 55.2, 3291 x 1528 x 6528 34.9 -> 36.1 /
    // 41.7 -> 37.2).  Fewer steps or rows: about even, or the halves (e4m3 1384 x 3888 x 1440 19.2 and 18.4 / 18.4 and 19.1, 352 x 16224 x 4768
    // 44.4 and 48.8 / 55.7 and 52.8, 145 x 22288 x 2528 23.1 and 24.2 / 28.8 and 30.4).  Of 26 sizes drawn at random the 11 that the rule
    // takes off the halves need 0.94 / 0.89 of their time on average, 1.03 / 0.98 at most, the 15 others would need 1.00 / 0.99.
    if (tail != 0 && 4 * tiles256 > cus && 2 * tiles256 <= cus)
      return ragged && M > 384 && (fp4 ? K / 2 : K) > 15 * kBK ? kSmallTiles : kTiles256Halves;
    if (tiles256 >= cus / 2) {
      // Whole rounds of the chip on 256 x 256 tiles; what is left over would keep the chip for another
      // full round however few tiles it is.  When its quadrants fit the chip at once it runs as
      // 128 x 128 quadrants instead: one round of those takes 0.5-0.6 of a round of tiles (measured on
      // MI355X, e4m3, us: 4096 x 5120 x 4096, 256 + 64 tiles, 97 -> 77; 4352^2 x 4096, 256 + 33, 97 -> 78;
      // 4096 x 4352 x 8192, 256 + 16, 177 -> 134; 6144^3, 512 + 64, 216 -> 186; 8448 x 8192^2, 1024 + 32,
      // 473 -> 436), two rounds of quadrants take as long as the round of tiles (4096 x 6144 x 4096,
      // 256 + 128: 97 -> 96).  Up to half a round of leftover tiles runs as 256 x 128 halves, a round of
      // which takes 0.8 of a round of tiles (the same shape 97 -> 87.5; 8192 x 5120 x 8192, 512 + 128,
      // 273 -> 258).  The results are the same bits either way.
      const int64_t left = tiles256 % cus;
      if (tail != 0 && tiles256 >= cus && left > 0 && cus % 8 == 0 && (tail >= 2 || 2 * left <= cus))
        return tail == 2 || (tail == 1 && 4 * left <= cus) ? kTiles256ThenQuads : kTiles256ThenHalves;
      return kTiles256;
    }
  }
  return kSmallTiles;
}

// The kernel for few tiles (mx_ring_kernels.hpp): tiles of 64 or 128 rows and columns, K shared between `splits` workgroups.
struct RingPlan {
  int tile_m, tile_n, splits;
  int64_t ns;  // what the estimate below gives, in nanoseconds
  int cols = 0;  // of the matrix that a tile covers, see ring_cols
};

// What a CU can have under way is what this kernel's time is made of, so the tiles and shares that a product takes
// follow from an estimate: a step costs 2 ns per line of 128 bytes that a workgroup asks for (a CU holds some 512
// requests, which take a microsecond from memory), or what its fragment reads and MFMAs take, and a workgroup about 2 us around
// its steps; sharing K costs the parked sums' way through memory.  The constants are a fit to 262 problems
// of 1 to 3712 rows, both operand types, K on and off a multiple of 128, and to 62 of 72 to 512 rows whose sizes are round, in each of up to 25
// forms, B from memory and from the memory-side cache: the form that the estimate picks takes 0.4 % longer than the best one of each
// problem on average (the round ones 0.8 %), 9 % at most (15 % for up to 64 rows).  A first fit, without the round ones, let shares
// of K cost 0.55 and 4 us where this has 0.8 and 6.7, and took 2.4 % longer on those, 41 % at most: 128 x 8192 x 8192 from the
// memory-side cache 23.9 -> 17.0 us, 384 x 1024 x 8192 15.5 -> 13.3.  On 57 others of
// 160 to 768 rows and round sizes it takes 0.7 % longer on average, 7 % at most.  `ragged`: the rows are not whole lines, a step more is on its way.
inline RingPlan plan_ring(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, size_t workspace_bytes, int cus, int split_k, int tile_m,
                          int tile_n) {
  const int64_t steps = ceil_div(fp4 ? K / 2 : K, (int64_t)kBK);
  const int64_t parked = workspace_bytes > kSplitTicketBytes ? (int64_t)(workspace_bytes - kSplitTicketBytes) : 0;
  RingPlan best{0, 0, 1, 0};
  for (int bm = 64; bm <= 128; bm += 64) {
    if (tile_m ? bm != tile_m : bm > 64 && M <= 64 && split_k <= 1) continue;  // (half a tile of rows that are not there is never the shorter one)
    for (int bn = 64; bn <= 128; bn += 64) {
      if (tile_n ? bn != tile_n : bn > 64 && N <= 64 && split_k <= 1) continue;
      const int64_t tiles = ceil_div(M, (int64_t)bm) * ceil_div(N, (int64_t)bn);
      const int area = bm * bn / 64;  // of 256
      const int lines = (int)std::min<int64_t>(M, bm) + (int)std::min<int64_t>(N, bn) + 8;
      const int step = std::max(2 * lines, 200 + 280 * area / 256), whole = 450 + 760 * (bm + bn) / 256;
      const auto consider = [&](int shares, int64_t ns) {
        if (best.tile_m == 0 || ns < best.ns) best = RingPlan{bm, bn, shares, ns};
      };
      const int extra = ragged ? 1 : 0;
      if (split_k <= 1 || tiles > (int64_t)(kSplitTicketBytes / 4))
        consider(1, whole + ceil_div(tiles, (int64_t)cus) * ((steps + extra) * step + 2200));
      if (tiles > (int64_t)(kSplitTicketBytes / 4) || split_k == 1) continue;
      // shares of six steps or more, a CU each; as many as asked for where that is said, if the workspace holds them
      const int t = (int)tiles, n = (int)steps, room = (int)std::min<int64_t>(parked / ((int64_t)bm * bn * 4 * t), kMaxSplits);
      const int most = std::min(room, split_k > 0 ? std::min(split_k, n) : std::min(std::min(cus / t, n / 6), kAutoMaxSplits));
      for (int splits = split_k > 0 ? std::max(most, 1) : 2; splits <= std::max(most, 1); ++splits) {
        const int per = (n + splits - 1) / splits, shares = (n + per - 1) / per, groups = t * shares;
        const int rounds = groups <= cus ? 1 : (groups + cus - 1) / cus;
        int64_t ns = whole + (int64_t)rounds * ((int64_t)(per + extra) * step + 2200);
        if (shares > 1) ns += 1250 + (800 * shares + 6700 * std::min(groups, cus) / cus) * area / 256;
        consider(shares, ns);
      }
    }
  }
  return best;
}

// Columns of the matrix that a tile covers.  Where whole tiles are one round and leave CUs without one, e4m3 tiles cover fewer, in eights: each CU asks for
// fewer lines, and B from memory that is what the launch's time is made of (us, whole tiles -> here: 200 x 5120 x 5120, 160 -> 256 tiles, 22.1 -> 18.0;
// 88 x 21328 x 8064, 167 -> 223, 50.2 -> 43.7; 358 x 3656 x 5120 22.1 -> 19.4).  From the memory-side cache the L2s' rate bounds it from some 180 workgroups on,
// and more of them ask for A more often (378 x 5840 x 10592 in 255 tiles 36.2 -> 40.2 us), so beyond those a tile stays wider than A's rows
// in it; and finding a tile's scales costs 0.2 us, so not where B is below 8 MiB (67 x 1288 x 1280 5.4 -> 5.1 from memory, 5.1 -> 5.3 from the cache).
// Of 130 products of 33 to 1500 rows drawn at random 25 change, to 0.94 / 1.00 of their time (geometric average, from memory / from the cache), where the others
// are at 0.98 / 0.99.  Not where K is shared (more is parked: 0.99 / 1.00, 1.09 at most), in several rounds (1022 x 4752 x 4928 44.8 -> 47.2) or
// for e2m1, whose scales come 16 bytes a lane (a word a lane costs 3 to 6 %, more than this gives).
inline int ring_cols(const RingPlan& p, bool fp4, int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t tiles_m = ceil_div(M, (int64_t)p.tile_m), tiles_n = ceil_div(N, (int64_t)p.tile_n);
  if (fp4 || p.splits > 1 || tiles_m * tiles_n > cus || K > ((int64_t)1 << 28) || N * K < ((int64_t)8 << 20)) return p.tile_n;  // (K: two chunks' scales in 32 bits)
  const auto for_tiles = [&](int64_t n) { return ceil_div(N, std::max(n / tiles_m, (int64_t)1)); };
  const int64_t rows = std::min(M, (int64_t)p.tile_m), cols = std::max(for_tiles(cus), std::min(for_tiles(cus * 17 / 24), rows + 8));
  const int fit = (int)std::max(std::min(ceil_div(cols, (int64_t)8) * 8, (int64_t)p.tile_n), (int64_t)p.tile_n / 2);
  return 8 * ceil_div(N, (int64_t)fit) >= 9 * tiles_n ? fit : p.tile_n;
}

// What the kernel of mx_few_rows.hip takes for a product of at most 64 rows, in nanoseconds.  Its workgroups walk whole rows of
// B, 16 or 32 columns each, with all of A beside them: per round of the chip 2.3 us, and per step and column 5.5 ns (5.2 off
// whole lines, where the rows do not begin on the same channels) and 1.6 ns per row of A.  columns: of a workgroup.
inline int64_t few_rows_ns(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, int cus, int columns) {
  const int64_t steps = ceil_div(fp4 ? K / 2 : K, (int64_t)kBK), rows = ceil_div(M, (int64_t)8) * 8;
  const int64_t rounds = ceil_div(ceil_div(N, (int64_t)columns), (int64_t)cus);
  return 1000 + 2260 * rounds + rounds * steps * (columns * (ragged ? 52 : 55) + 16 * rows) / 10 - 8 * rows;
}

// The kernel for at most 32 rows by whole lines (mx_few_lines_kernels.hpp): octets of columns per group, and what the estimate gives in nanoseconds.
struct FewLinesPlan {
  int octets;
  int64_t ns;
};

// Per round of the chip a workgroup's turns along K take what its waves take for one, or 2.3 ns per line that they ask for, and all
// rounds together no less than B at 5.7 TB/s; per group the sums' way through LDS.  The constants are a fit to 161 problems of 1 to 32 rows, 512 to 28672
// columns and K of 512 to 16384, both operand types, on and off whole lines, in all eight forms each, to the geometric mean of the time with B from memory and from
// the memory-side cache: the form that it picks takes 0.3 % longer than the best one of each problem from memory and 0.7 % from the cache.  What it is held against is
// 2 % more, 10 % for e4m3 off whole lines: of 799 problems of 1 to 32 rows, most of them where small tiles are close, the choice between the two then takes 0.18 % longer
// than the shorter one (geometric mean of both; 0.51 % without it, with 22 problems more than 8 % longer instead of 6), e4m3 2 x 16904 x 1120 by lines 9.9 / 7.0 and
// small tiles 8.2 / 5.9 us, 18 x 1480 x 15328 15.9 / 11.4 and 12.2 / 10.6.
inline FewLinesPlan plan_few_lines(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, int cus, int octets) {
  const int64_t k_bytes = fp4 ? K / 2 : K, steps = ceil_div(k_bytes, (int64_t)kBK);
  const int mh = (int)((M + 7) / 8), rows_tiles = (mh + 1) / 2;
  FewLinesPlan best{0, 0};
  for (int nh = octets ? octets : 1; nh <= (octets ? octets : 8); ++nh) {
    const int waves = few_lines_waves(fp4, mh, nh, ragged), tiles = rows_tiles * ((nh + 1) / 2);
    const int64_t rounds = ceil_div(few_lines_groups(N, nh), (int64_t)cus), turns = ceil_div(steps, (int64_t)waves) + (ragged ? 1 : 0);
    const int64_t turn = std::max<int64_t>(386 + 11 * tiles * (fp4 ? 2 : 1), waves * (8 * nh + M + 4) * 227 / 100);
    const int64_t ns = 1770 + rounds * (125 + 190 * tiles) + std::max(rounds * turns * turn, N * k_bytes * 10 / 57000);
    if (!best.octets || ns < best.ns) best = FewLinesPlan{nh, ns};
  }
  best.ns = best.ns * (ragged && !fp4 ? 110 : 102) / 100;
  return best;
}

// Which of the two kernels a product of at most 32 rows is for: the one of mx_few_rows.hip keeps the short rows of few columns that are no whole lines,
// a workgroup of 16 columns per CU at most.  A wave by whole lines asks for a window more than it has steps there, and reads a step's fragments out of two;
// the other one has 16 steps of at most 16 rows in its waves' first turn (us, by whole lines and there, from memory / from the
// memory-side cache: e2m1 32 x 280 x 544 3.42 / 3.67 and 2.77 / 3.00, 19 x 2520 x 1344 3.90 / 3.72 and 3.47 / 3.12, 30 x 2368 x 4576 7.05 / 5.97 and 6.64 / 4.65,
// 4 x 3872 x 2720 4.78 / 3.88 and 4.71 / 3.28, e4m3 25 x 400 x 320 3.16 / 3.33 and 2.81 / 2.95, 1 x 3168 x 1120 4.19 / 3.61 and 4.08 / 3.23).  Of 519 problems
// of 1 to 32 rows drawn at random, half of them on whole lines, none of these is faster there by more than 3 %, and beyond these limits none
// by more than 7 %.
inline bool few_rows_instead_of_lines(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, int cus) {
  const int64_t steps = ceil_div(fp4 ? K / 2 : K, (int64_t)kBK);
  if (!ragged || N > 16 * (int64_t)cus) return false;
  return steps <= (fp4 && M > 16 ? 24 : 16) && (fp4 || M > 16 || steps > 8);
}

struct GemmKnobs {  // gemm.variant, gemm.tail_quads, gemm.split_k, gemm.tile_m, gemm.tile_n, gemm.few_rows_octets
  int variant, tail, split_k, tile_m, tile_n, octets = 0;
};
struct GemmPlan {
  GemmTiles tiles;
  RingPlan small;  // of kSmallTiles
  FewLinesPlan lines = {};  // of kFewLines
};

// K counts elements; ragged: see ring_ragged; workspace_bytes 0: none; few_columns: columns of B that a workgroup of the kernel for at most 64 rows
// takes, 0 where it cannot take the product; few_lines: whether the one for at most 32 can, which then stands in its place unless
// few_rows_instead_of_lines.
// Either is taken where it needs less time than the small tiles.  Those read B at 4.8 TB/s from memory at most, and at 6.5 to 7.3 from the memory-side cache: the
// first is also taken where it needs less than reading B at 4.8 TB/s, the second than at 5.2, which is in between (us, small tiles and by
// whole lines, 16 x 28672 x 4096 28.0 / 19.5 and 22.8 / 19.5; with 4.8 here 18 x 21728 x 8992 is lost, 38.4 / 30.1 and 40.2 / 36.7).
// (33 to 64 rows: fitted to 150 problems of 1 to 64 rows, and off whole lines to 340: at 350 others of 128 to 12000 columns drawn at random, half of them of
// few columns and a long K, where the choice is close, what the two estimates pick takes 0.2 % longer than the better kernel with B from memory,
// 13 % at most, and 1.0 % from the memory-side cache, 25 % at most, where few rows gain more.  With 6.6 ns off whole lines these were 0.25 %
// and 1.7 %, 50 % at most: e2m1 12 x 1488 x 12064 from the cache 8.9 and 6.9 us, 1 x 168 x 10048 7.6 and 5.1, from memory 7.9 and 6.4.
// A rule on sizes, few rows for K of 2048 and N of 1024 on with exceptions, took 27 % longer on the 150.
// Up to 32 rows: of the 161 problems that plan_few_lines is fitted to, what the estimates pick takes 1.2 / 2.2 % longer than the best of the three kernels
// (from memory / from the cache), and 0.91 / 0.91 of what it took without the kernel by whole lines.  What that one lost to the other one for few
// rows stays with it.)
// How many workgroups are to share K does not decide between the two; whether any may does.
inline GemmPlan plan_gemm(bool fp4, int64_t M, int64_t N, int64_t K, bool ragged, size_t workspace_bytes, int cus, int few_columns, bool few_lines,
                          GemmKnobs knobs) {
  const auto small = [&](int split_k, int tile_m, int tile_n) {
    GemmPlan p{kSmallTiles, plan_ring(fp4, M, N, K, ragged, workspace_bytes, cus, split_k, tile_m, tile_n)};
    p.small.cols = ring_cols(p.small, fp4, M, N, K, cus);
    return p;
  };
  if (knobs.variant == 1) return small(knobs.split_k, 128, 128);
  if (knobs.variant == 3) return small(knobs.split_k, knobs.tile_m, knobs.tile_n);
  if (few_columns && knobs.variant == 10) return {kFewRows, {}};
  if (few_columns && (knobs.variant == 9 || knobs.variant == 0)) {
    GemmPlan few{kFewRows, {}};
    int64_t few_ns = 0;
    const bool by_lines = few_lines && (knobs.octets || !few_rows_instead_of_lines(fp4, M, N, K, ragged, cus));
    if (by_lines) {
      few = {kFewLines, {}, plan_few_lines(fp4, M, N, K, ragged, cus, knobs.octets)};
      few_ns = few.lines.ns;
    } else {
      few_ns = few_rows_ns(fp4, M, N, K, ragged, cus, few_columns);
      if (few_ns < 3000 + N * (fp4 ? K / 2 : K) / 4800) return few;
    }
    if (knobs.variant == 9) return few;
    const GemmPlan tiles = small(knobs.split_k == 1 ? 1 : 0, 0, 0);
    if (few_ns < std::max(tiles.small.ns, by_lines ? 2700 + N * (fp4 ? K / 2 : K) / 5200 : 0)) return few;
    return knobs.split_k > 1 ? small(knobs.split_k, 0, 0) : tiles;
  }
  const GemmTiles tiles = plan_tiles(fp4, M, N, K, ragged, cus, knobs.variant, knobs.tail);
  return tiles == kSmallTiles ? small(knobs.split_k, 0, 0) : GemmPlan{tiles, {}};
}

}  // namespace dt
