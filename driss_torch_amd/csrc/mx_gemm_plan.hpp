// Which kernel a block-scaled product of more rows than the few-rows kernel takes runs on, and how many
// workgroups share a tile's K: plain arithmetic on sizes, without the device.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "dt_host.hpp"

namespace dt {

constexpr int kBK = 128;             // K bytes per step = one 16x16x128 MFMA
constexpr size_t kSplitTicketBytes = 1024;        // head of the split-K workspace: one counter per 128 x 128 tile
constexpr size_t kSplitTileBytes = 128 * 128 * 4;  // parked fp32 accumulators of one tile and split
constexpr int kMaxSplits = 16;      // what gemm.split_k may force
constexpr int kAutoMaxSplits = 12;  // what the library picks by itself

// Split-K factor for the 128 x 128 tiling.  A grid of half a workgroup per CU or less leaves
// most of the chip idle while each workgroup walks the whole K, one K-step per memory latency / 3:
// share K between as many workgroups per tile as fill the chip once.  What it costs is the last
// workgroup of a tile reading every share through one CU (about 1 us per share of a full tile),
// so shares are 16 K-steps on average or more, or 10 while there are at most four shares of a K of 5120 elements
// or more (the last one is what is left: 41 steps are shared 11 + 11 + 11 + 8;
// measured on MI355X, e4m3, B rotated through memory, us without -> with: 16 x 8192 x 8192 31 -> 19,
// 128 x 8192 x 8192 42 -> 24, 1024 x 1024 x 16384 58 -> 34, 512 x 512 x 65536 219 -> 50, 128 x 128 x 16384
// 56 -> 25, 128 x 5120 x 5120 with four shares of 10 steps 19.9 -> 17.5, with six 19.4, 256 x 5120 x 5120 with
// three 22.7 -> 19.9, 256 x 4096 x 4096 with three 15.7 -> 16.4; e2m1 128 x 8192 x 8192 with three 24.5 -> 18.2).
// Two shares pay where they fill four fifths of the chip or more and save more steps than the 8 us that
// parking and adding a whole chip's tiles takes: from 56 steps on, or 32 when B comes from memory and each
// step takes longer (256 x 8192 x 8192 41 -> 33, 512 x 4096 x 14336 69 -> 46, 128 x 14336 x 4096 24.8 -> 22.6;
// not 1000 x 2048 x 6144 23.0 -> 25.4, 128 x 5120 x 5120 19.9 -> 22.1, nor e2m1 96 x 14336 x 4096 14.7 -> 16.0). The knob
// gemm.split_k forces a factor (1 = never split); whatever is asked for, every split owns a step
// and the workspace holds all shares.
inline int plan_splits(bool fp4, int64_t M, int64_t N, int64_t k_steps, size_t workspace_bytes, int cus, int forced) {
  const int64_t tiles = ceil_div(M, 128) * ceil_div(N, 128);
  if (workspace_bytes <= kSplitTicketBytes || tiles > (int64_t)(kSplitTicketBytes / 4)) return 1;
  const int64_t room = (int64_t)((workspace_bytes - kSplitTicketBytes) / kSplitTileBytes) / tiles;
  int64_t want;
  if (forced > 0) {
    want = forced;
  } else {
    const int64_t shares = std::max(k_steps * (fp4 ? 2 : 1) >= 40 ? std::min<int64_t>(k_steps / 10, 4) : 0, k_steps / 16);
    want = cus / tiles;
    if (want > shares) want = shares;
    if (want > kAutoMaxSplits) want = kAutoMaxSplits;
    const bool two_pay = tiles * 5 >= cus * 2 && (k_steps >= 56 || (k_steps >= 32 && N * k_steps * kBK >= ((int64_t)32 << 20)));
    if (want < 2 || (want == 2 && !two_pay)) return 1;
  }
  if (want > kMaxSplits) want = kMaxSplits;
  if (want > room) want = room;
  if (want > k_steps) want = k_steps;
  if (want < 2) return 1;
  const int64_t per = ceil_div(k_steps, want);
  return (int)ceil_div(k_steps, per);
}

enum GemmTiles {
  kTiles128,                 // 128 x 128, with K shared where splits > 1
  kTiles256Halves,           // 256 x 128 halves of 256 x 256 tiles
  kTiles256x192,
  kTiles256,
  kTiles256ThenQuads,        // whole rounds of 256 x 256, the tiles left over as 128 x 128 quadrants
  kTiles256ThenHalves,       // or as halves
  kTiles256QuadrantSchedule  // 256 x 256 on the other tiles' main loop (on request only)
};
struct GemmPlan {
  GemmTiles tiles;
  int splits;  // workgroups that share K per tile (kTiles128)
};

// K counts elements; workspace_bytes 0: none.  variant, tail, split_k: the knobs gemm.variant, gemm.tail_quads
// and gemm.split_k.
inline GemmPlan plan_gemm(bool fp4, int64_t M, int64_t N, int64_t K, size_t workspace_bytes, int cus, int variant, int tail,
                          int split_k) {
  const int64_t tiles256 = ceil_div(M, 256) * ceil_div(N, 256);
  // 256 x 192 tiles where they fill the chip's one round better than 256 x 256 tiles do (which leave a
  // quarter of it idle or more).  At the chip's power limit a round of them takes 0.78 of a round of the
  // large tiles, not 0.75, so they only pay while both are one round (us, 256 x 256 -> 256 x 192, e4m3 and
  // e2m1: 2048 x 4352 x 4096, 136 -> 184 tiles, 38.5 -> 34.3 and 26.0 -> 23.6; 2048 x 5120 x 5120, 160 -> 216,
  // 48.3 -> 45.3 and 30.9 -> 29.3; 2000 x 6144 x 8192, 192 -> 256, 80.0 -> 77.7 and 50.9 -> 49.2; two rounds
  // against one and a half: 4096 x 5632 x 4096 77.9 and 77.9, 4096 x 9216 x 4096 120.9 -> 123.5).
  const int64_t tiles192 = ceil_div(M, 256) * ceil_div(N, 192);
  if (variant == 5 || (variant == 0 && 2 * tiles256 > cus && tiles192 > tiles256 && tiles192 <= cus)) return {kTiles256x192, 1};
  if (variant == 2) return {kTiles256, 1};
  if (variant == 7) return {kTiles256QuadrantSchedule, 1};
  // One round of 128 x 128 tiles is taken before anything larger.  Between a quarter and half a round of
  // 256 x 256 tiles: as 256 x 128 halves they fill the chip once (0.8 of a round of tiles), as 128 x 128 tiles
  // two rounds (2 x 0.55) unless rows or columns past the matrix leave much of the large tiles idle.  With at
  // most 128 rows (or an odd number of 128-row bands) that may be one round, which is the shorter one then, also
  // at exactly half a round of the large tiles (us, halves -> 128 x 128, e4m3 and e2m1: 96 x 28672 x 4096
  // 34.6 -> 30.6 and 21.4 -> 16.9, 128 x 32768 x 4096 39.5 -> 35.7 and 24.9 -> 19.3 where 256 x 256 tiles take 53.1
  // and 32.3, 1152 x 3584 x 4096 26.4 -> 22.7 and 19.3 -> 15.9).
  if (variant == 0 && ceil_div(M, 128) * ceil_div(N, 128) > cus) {
    if (tail != 0 && 4 * tiles256 > cus && 2 * tiles256 <= cus) return {kTiles256Halves, 1};
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
        return {tail == 2 || (tail == 1 && 4 * left <= cus) ? kTiles256ThenQuads : kTiles256ThenHalves, 1};
      return {kTiles256, 1};
    }
  }
  return {kTiles128, plan_splits(fp4, M, N, ceil_div(fp4 ? K / 2 : K, (int64_t)kBK), workspace_bytes, cus, split_k)};
}

}  // namespace dt
