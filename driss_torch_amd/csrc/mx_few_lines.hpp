// The block-scaled GEMM for at most 32 rows by whole lines of B (mx_few_lines_kernels.hpp): what the dispatch needs of it, and
// which of its forms a product takes.  Plain arithmetic on sizes, without the device.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dt_host.hpp"

namespace dt {

// B's rows (output columns) come in octets of eight, in the order of their scales: a 512-byte chunk holds the scale words of 128 rows, the eight
// of octet 4 q + b (rows 32 b + 8 q to 32 b + 8 q + 7) in word b of its lines 8 q to 8 q + 7, so that four octets in a row share 128 bytes of them.
__host__ __device__ inline uint32_t octet_column(uint32_t octet) { return (octet >> 4) * 128u + (octet & 3u) * 32u + ((octet >> 2) & 3u) * 8u; }

// The scale word of a row of an octet, in its chunk
__host__ __device__ inline uint32_t octet_scale_word(uint32_t octet, uint32_t row) { return ((octet >> 2) & 3u) * 128u + row * 16u + (octet & 3u) * 4u; }

// Groups of `octets` octets each that hold a column of the matrix.
inline int64_t few_lines_groups(int64_t N, int octets) {
  const int64_t whole = N / 128 * 16, rest = N % 128;
  int64_t last = whole;  // one past the last octet with a column
  for (int o = 0; o < 16; ++o)
    if (octet_column((uint32_t)o) < (uint32_t)rest) last = whole + o + 1;
  return ceil_div(last, (int64_t)octets);
}

// A wave's ring in LDS: stages of a K-step's lines of its operands and their scale words, whole tiles of 16 rows.
constexpr int kFewLinesLds = 160 * 1024;
constexpr bool few_lines_scales_in_one(int mh, int nh) { return mh <= 4 && nh <= 4; }  // 32 words of B and 32 of A, one load
constexpr int few_lines_scale_loads(bool fp4, int mh, int nh) { return (fp4 ? 2 : 1) * (few_lines_scales_in_one(mh, nh) ? 1 : 2); }
constexpr int few_lines_loads(bool fp4, int mh, int nh) { return nh + mh + few_lines_scale_loads(fp4, mh, nh); }
constexpr int few_lines_stage(bool fp4, int mh, int nh) {
  return (nh + nh % 2 + mh + mh % 2) * 1024 + few_lines_scale_loads(fp4, mh, nh) * 256;
}
// Stages with `waves` waves in a workgroup: what fits the LDS, the 6 bits of the counter of loads and the 16 of an LDS instruction's offset
constexpr int few_lines_stages_of(int waves, bool fp4, int mh, int nh) {
  int s = kFewLinesLds / waves / few_lines_stage(fp4, mh, nh);
  while ((s - 1) * few_lines_loads(fp4, mh, nh) > 63 || s * few_lines_stage(fp4, mh, nh) > 65536) --s;
  return s;
}
// Waves that share K: eight for the narrowest groups (products of few columns, whose time is a wave's turns), else four, or two where four would
// have no stage under way besides those in use (us, four waves -> eight, from memory / from the memory-side cache: groups of two octets, e4m3 23 x 2344 x 2848
// 5.2 -> 4.9 / 4.9 -> 4.3; of four, 6 x 3072 x 2048 4.1 -> 3.8 / 3.6 -> 3.3, but 16 x 8192 x 8192 14.4 -> 15.5 / 12.9 -> 13.9)
constexpr int few_lines_waves(bool fp4, int mh, int nh, bool ragged) {
  const int least = ragged ? 4 : 3;
  if (nh <= 2 && few_lines_stages_of(8, fp4, mh, nh) >= 3) return 8;
  return few_lines_stages_of(4, fp4, mh, nh) >= least ? 4 : 2;
}

// Whole lines of B go out in runs of four loads: load i of an octet's eight rows has i % 4 KiB as its immediate offset, which counts in memory and in LDS, so its
// lane offsets are lowered by as much.  Octets are not in the order of their columns (load 3 may be column 8 of its chunk, and a column that is not there is the
// last one, in front of that), so with rows of a few lines the lowered offset of a byte can lie in front of the chunk: B's descriptor begins
// kFewLinesBias bytes in front of it, and no lane offset depends on how a sum below zero is taken.
constexpr uint32_t kFewLinesBias = 3 * 1024;
constexpr uint32_t few_lines_immediate(int load) { return (uint32_t)(load % 4) * 1024u; }
__host__ __device__ inline uint32_t few_lines_lane_offset(uint32_t row, uint32_t ldb, uint32_t in_row, int load) {
  return kFewLinesBias + row * ldb + in_row - few_lines_immediate(load);
}
// The row of B, from the group's first chunk on, that lane octet row lrow of load i brings: a column that is not there reads the last one's bytes
__host__ __device__ inline uint32_t few_lines_row(uint32_t first_octet, int i, uint32_t lrow, uint32_t rows) {
  const uint32_t r = octet_column(first_octet + i) - (first_octet >> 4) * 128u + lrow;
  return r < rows ? r : rows - 1u;
}

// What the kernel takes: scale chunks of up to 4 K bytes in 32 bits
inline bool few_lines_fits(int64_t M, int64_t K) { return M <= 32 && K <= ((int64_t)1 << 29); }

// What the knobs gemm.few_rows_octets and gemm.few_rows_tiles (two octets each) ask for, 0: what the estimate picks.
inline int few_lines_forced_octets() {
  const int octets = tuning(Knob::gemm_few_rows_octets), tiles = tuning(Knob::gemm_few_rows_tiles);
  return octets >= 1 && octets <= 8 ? octets : tiles == 1 || tiles == 2 ? 2 * tiles : 0;
}

struct FewLinesArgs {  // operands as for dt_mx_fp8_bf16 / dt_mx_fp4_bf16, already checked; M <= 32
  const uint8_t *a, *b, *sfa, *sfb;
  int64_t M, N, K, lda, ldb;
  void* out;
  int64_t ldo;
  hipStream_t stream;
};
// octets: 1 to 8 per group; ragged: rows that are no whole lines or do not begin on one (ring_ragged).  Returns a dt_status.
int launch_few_lines_e4m3(const FewLinesArgs& p, bool ragged, int octets);
int launch_few_lines_e2m1(const FewLinesArgs& p, bool ragged, int octets);

}  // namespace dt
