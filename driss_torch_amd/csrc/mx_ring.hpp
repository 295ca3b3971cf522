// The block-scaled GEMM for few tiles (mx_ring_kernels.hpp): what the dispatch needs of it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dt {

struct RingArgs {  // operands as for dt_mx_fp8_bf16 / dt_mx_fp4_bf16, already checked
  const uint8_t *a, *b, *sfa, *sfb;
  int64_t M, N, K, lda, ldb;
  void* out;
  int64_t ldo;
  void* workspace;
  hipStream_t stream;
  int cols;  // of the matrix that a tile covers (ring_cols)
};

// Rows that are no whole lines of 128 bytes, or do not begin on one: the kernel's form that deals with it.
inline bool ring_ragged(int64_t k_bytes, const uint8_t* a, const uint8_t* b, int64_t lda, int64_t ldb) {
  return k_bytes % 128 != 0 || lda % 128 != 0 || ldb % 128 != 0 || reinterpret_cast<uintptr_t>(a) % 128 != 0 || reinterpret_cast<uintptr_t>(b) % 128 != 0;
}

// Tiles of tile_m x tile_n (64 or 128 each), K shared between `splits` workgroups per tile.  Returns a dt_status.
int launch_ring_e4m3(const RingArgs& p, bool ragged, int tile_m, int tile_n, int splits);
int launch_ring_e2m1(const RingArgs& p, bool ragged, int tile_m, int tile_n, int splits);

// What the kernel's loads ask for.  A load goes through a buffer descriptor (base, number of bytes) with an offset per lane, an immediate
// and a scalar one; one past the end reads nothing.  Whether the scalar offset counts there is left open here: a load past the end is past
// it by its lane offset alone, and an empty descriptor goes with a scalar offset of zero.

// A descriptor and the scalar offset into it for one window along K; nothing past the last window.
struct RingAsk {
  uint32_t bytes, at;
};
__host__ __device__ inline RingAsk ring_ask(bool in, uint32_t bytes, uint32_t at) { return in ? RingAsk{bytes, at} : RingAsk{0u, 0u}; }

// The scales of a tile, `chunks` times 512 bytes: 512 bytes a K-step (e4m3; waves of even and odd number bring half of them each) or 1024.  The
// descriptor ends with the last step of the share, or with the last chunk where K ends in the middle of that step.
__host__ __device__ inline uint32_t ring_scale_bytes(bool fp4, int chunks, int end_step) {
  const int end = end_step * (fp4 ? 2 : 1);
  return (uint32_t)(end < chunks ? end : chunks) * 512u;
}
__host__ __device__ inline uint32_t ring_scale_offset(bool fp4, int wave, int lane, int step) {
  return (uint32_t)step * (fp4 ? 1024u : 512u) + (fp4 ? lane * 16u : (wave & 1) * 256u + lane * 4u);
}
// What is added to that for e4m3 where a tile begins anywhere in a chunk: word `word` of the 128 that go to LDS is that of the tile's row
// t = word % 4 * 32 + word / 4 (rows past the tile: the last one's), which lies in the chunk of row0 or in the next one of the matrix, so the
// descriptor spans both.
__host__ __device__ inline uint32_t ring_scale_shift(int row0, int rows, int chunks, int word) {
  const int t = (word & 3) * 32 + (word >> 2), r = row0 + (t < rows ? t : rows - 1);
  return (uint32_t)((r >> 7) - (row0 >> 7)) * ((uint32_t)chunks * 512u) + (uint32_t)((r & 31) * 16 + ((r >> 5) & 3) * 4 - word * 4);
}
__host__ __device__ inline uint32_t ring_scale_span(int row0, int rows, int chunks) {
  return (uint32_t)(((row0 + rows - 1) >> 7) - (row0 >> 7)) * ((uint32_t)chunks * 512u);
}

// A panel of up to 128 rows, from one step along K on: `left` bytes of each row.  mis: bytes from the descriptor's base, a multiple of 128, to
// the first of them (RAGGED; whole lines: 0).
struct RingPanel {
  uint32_t mis;
  int rows, left;
  int64_t ld;
  __host__ __device__ uint32_t bytes() const { return (uint32_t)((rows - 1) * ld + left + mis); }
  // offset of a lane's 16 bytes of row r in window 0: lane L brings row L / 8 of a group of eight, and its chunk L % 8 turned by the row and by how
  // far into a line it begins.  Rows past the matrix (whole lines): further than any descriptor reaches, as 255 rows span less than 4 GiB and a
  // panel has 128.  (A select, not a branch: around four branches the compiler loads the kernel's arguments later, 0.25 us a launch.)
  __host__ __device__ uint32_t start(bool ragged, int r, int lane) const {
    const int lrow = lane >> 3;
    const uint32_t phase = ragged ? (mis + (uint32_t)lrow * (uint32_t)ld) & 127u : 0u;
    const uint32_t chunk = ((lane & 7) - lrow + (phase >> 4)) & 7u;
    const uint32_t here = mis + (uint32_t)r * (uint32_t)ld - phase + chunk * 16u, nowhere = 0xF0000000u + chunk * 16u;
    return !ragged && r >= rows ? nowhere : here;
  }
  // RAGGED: the row's last 16 bytes; a lane never asks for anything behind them (rows past the matrix: past the descriptor's end)
  __host__ __device__ uint32_t end(int r) const { return mis + (uint32_t)r * (uint32_t)ld + left - 16; }
};

}  // namespace dt
