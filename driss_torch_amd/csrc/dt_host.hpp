// Host-side helpers shared by the C-ABI entry points: argument checks, device facts,
// the workspace layout and the tuning table.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "driss_torch_hip.h"

namespace dt {

// ---- workspace layout (see dt_workspace_bytes in the public header) -----------------
constexpr int kMaxPartials = 8192;          // upper bound on the grid of a reduction kernel
constexpr size_t kWsTicket = 0;             // u32 arrival counter, zero between launches
constexpr size_t kWsRunning = 128;          // u32 running max of |x| bits, zero between launches
constexpr size_t kWsAmax = 64;              // f32 amax of the last reduction
constexpr size_t kWsScale = 68;             // f32 scale[2] derived from it
constexpr size_t kWsPartials = 3072;        // u32 maxima of a reduction's workgroups, for the cast behind it
constexpr int kWsPartialWords = 256;
constexpr size_t kWsBytes = 4096;

struct DeviceFacts {
  int cu_count;
};
const DeviceFacts& device_facts();  // of the current device, cached per device

// Launch-shape knobs.  Workgroups per CU for the persistent grids, chosen on MI355X.
//   dynamic.resident: 1 = per-tensor dynamic quantization of a tensor that fits the chip runs as one
//                 kernel that keeps it in registers and LDS.  That kernel waits inside for all of its
//                 workgroups and so assumes that this process has the GPU to itself: 0 unless the caller
//                 opts in (dt_set_exclusive_gpu, or DRISS_TORCH_RESIDENT=1 in the environment when the
//                 library is loaded); dynamic.resident_min_kib = smallest such
//                 tensor (-1: as measured, 58 MiB, of 16-bit tensors to both types 52); sizes in [resident_gap_lo_kib, resident_gap_hi_kib) take the two kernels
//                 dynamic.resident_overflow: 1 = tensors of up to 4 x the chip's capacity keep what fits
//                 and read only the rest twice
//   amax.blocks_per_cu: most workgroups per CU of a reduction in workgroups of 256 or 512 threads (those of 1024 are at
//                 most five per eight CUs whatever it says)
//   rowwise.block_from_vecs: rows of at least this many 16-byte vectors get a workgroup each (shorter
//                 ones a wave each)
//   mx.dual:      1 = dt_mx_fp8_quantize_dual reads x once (0: two single casts)
//   mx.colt_via_dual: 1 = the transposed column cast runs as the one-read kernel without its row half
//   mx.dual_order: tile order of the one-read kernel: -1 = chosen by shape, 0 = down the rows first, 1 = along
//                 the columns first, 2 = bands of 8 row tiles
//   mx.dual_narrow: its tiles: -1 = chosen by shape, 0 = wide (256 columns of 16 bits, 128 of fp32), 1 = half as wide (fp32: columns alone)
//   mx.colt_pipe: the transposed column cast as a grid of this many workgroups per CU that walk the tiles
//                 with the next tile's loads in flight (0 = one workgroup per tile)
//   mx.row_band4: 1 = row-wise MX cast with blocked scales walks 4 rows x 512 elements per wave pass
//   gemm.variant: 0 = pick the tile by problem size, 1 = 128x128 tiles, 2 = 256x256 tiles, 3 = tiles of 64 or 128 rows
//                 and columns as gemm.tile_m and gemm.tile_n say (0 = by the estimate), 5 = 256x192 tiles,
//                 7 = 256x256 tiles on the main loop of the smaller ones (quadrants of the wave tile, no L2 prefetch;
//                 the same bits), 9 = the kernels for at most 64 rows whatever the other dimensions, 10 = the one that loads B into registers
//                 (mx_few_rows.hip) whichever of them the rule takes
//   gemm.few_rows_tiles: 16-column tiles per group of columns of those kernels: 0 = by the problem's size, 1, 2
//   gemm.few_rows_per_cu, gemm.few_rows_stagger, gemm.few_rows_steps: of the one that loads B into registers, workgroups per CU (0: two), the
//                 staggered walk along K, steps per batch of loads (0: two for at most 16 rows, else one; 1, 2: up to 32 rows)
//   gemm.few_rows_octets: columns per group of the one for at most 32 rows, in eights: 0 = by the problem's size, 1 to 8
//   gemm.tail_quads: 1 = tiles left over after whole rounds of 256x256 tiles run as 128x128 quadrants
//                 or 256x128 halves when those fit the chip at once, 0 = never, 2 = always as
//                 quadrants, 3 = always as halves
//   gemm.split_k: of the small tiles, 0 = share K between workgroups when they leave CUs idle (needs the
//                 workspace of the _ws entry points), 1 = never, n = n workgroups per tile
#define DT_KNOBS(X) \
  X(gemm, few_rows_tiles, 0)               \
  X(gemm, few_rows_stagger, 1)             \
  X(gemm, few_rows_steps, 0)               \
  X(gemm, few_rows_per_cu, 0)              \
  X(gemm, few_rows_octets, 0)              \
  X(amax, blocks_per_cu, 1)                \
  X(amax, stream_before_cast, 0)           \
  X(cast, blocks_per_cu, 0)                \
  X(cast, unroll, 0)                       \
  X(cast, pair_blocks_per_cu, 0)           \
  X(rowwise, block_from_vecs, 257)         \
  X(mx, blocks_per_cu, 32)                 \
  X(mx, col_blocks_per_cu, 32)             \
  X(mx, dual, 1)                           \
  X(mx, dual_order, -1)                    \
  X(mx, dual_narrow, -1)                   \
  X(mx, colt_pipe, 2)                      \
  X(mx, colt_via_dual, 1)                  \
  X(mx, row_band4, 1)                      \
  X(gemm, variant, 0)                      \
  X(gemm, tile_m, 0)                       \
  X(gemm, tile_n, 0)                       \
  X(gemm, split_k, 0)                      \
  X(gemm, tail_quads, 1)                   \
  X(dynamic, resident, 0)                  \
  X(dynamic, resident_min_kib, -1)         \
  X(dynamic, resident_gap_lo_kib, 0)       \
  X(dynamic, resident_gap_hi_kib, 0)       \
  X(dynamic, resident_overflow, 1)         \
  X(dynamic, resident_spin_limit, 1 << 19)

enum class Knob : int {
#define DT_KNOB_ID(group, name, value) group##_##name,
  DT_KNOBS(DT_KNOB_ID)
#undef DT_KNOB_ID
  count
};
// Set from any thread while launches on other threads read them.  A launch reads several: by their place in the
// list (by name, as dt_set_tuning finds them, one cost a launch 50 to 100 ns).
extern std::atomic<int> g_knob_values[];
inline int tuning(Knob k) { return g_knob_values[(int)k].load(std::memory_order_relaxed); }

// Per-workgroup clock readings for the benchmark's phase report exist only in a build with
// -DDT_PHASE_LOG (a second library made for that report); in the product build kPhaseLog is false, the
// kernels' stamps compile to nothing and the entry point that sets the buffer is not there.
#ifdef DT_PHASE_LOG
constexpr bool kPhaseLog = true;
// Device buffer for the readings (dt_set_phase_log), or null when none is set, it holds fewer than
// `need_bytes`, or it lives on another device than the current one.
uint64_t* phase_log(size_t need_bytes);
#else
constexpr bool kPhaseLog = false;
inline uint64_t* phase_log(size_t) { return nullptr; }
#endif

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int64_t ceil_div(int64_t a, int64_t b) { return a / b + (a % b != 0); }  // src/include/utils.h:37-39

// launcher(kernel, grid, block, lds, stream)(arguments...): what kernel<<<grid, block, lds, stream>>>(arguments...) does, without its detour by a
// call configuration that is stored and fetched again, 2.38 against 2.60 us of the host per launch.  A failure is the last error (launch_status).
template <typename... P>
struct Launcher {
  void (*kernel)(P...);
  unsigned grid, block;
  size_t lds;
  hipStream_t stream;
  void operator()(P... arguments) const {
    void* at[] = {&arguments...};
    (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(block), at, lds, stream);
  }
};
template <typename... P>
inline Launcher<P...> launcher(void (*kernel)(P...), unsigned grid, unsigned block, size_t lds, hipStream_t stream) {
  return {kernel, grid, block, lds, stream};
}

inline int launch_status() { return hipGetLastError() == hipSuccess ? DT_OK : DT_ERR_LAUNCH; }

inline hipStream_t as_hip(dt_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace dt
