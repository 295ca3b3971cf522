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
};

// Rows that are no whole lines of 128 bytes, or do not begin on one: the kernel's form that deals with it.
inline bool ring_ragged(int64_t k_bytes, const uint8_t* a, const uint8_t* b, int64_t lda, int64_t ldb) {
  return k_bytes % 128 != 0 || lda % 128 != 0 || ldb % 128 != 0 || reinterpret_cast<uintptr_t>(a) % 128 != 0 || reinterpret_cast<uintptr_t>(b) % 128 != 0;
}

// Tiles of tile_m x tile_n (64 or 128 each), K shared between `splits` workgroups per tile.  Returns a dt_status.
int launch_ring_e4m3(const RingArgs& p, bool ragged, int tile_m, int tile_n, int splits);
int launch_ring_e2m1(const RingArgs& p, bool ragged, int tile_m, int tile_n, int splits);

}  // namespace dt
