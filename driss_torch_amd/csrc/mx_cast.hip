// dt_mx_fp8_quantize / dt_to_blocked: MXFP8 cast with E8M0 block-32 scales (C ABI).
#include "mx_cast_plan.hpp"
#include "mx_kernels.hpp"

namespace {
using namespace dt;

// The general kernel writes scale bytes one by one and no padding: the blocked buffer starts out as zeros
int zero_blocked_padding(uint8_t* scale, int64_t SR, int64_t SC, hipStream_t s) {
  if (SR % 128 == 0 && SC % 4 == 0) return DT_OK;  // the cast writes every byte
  const int64_t n = dt_blocked_scale_bytes(SR, SC);
  launcher(fill_bytes_kernel, (unsigned)std::min<int64_t>(ceil_div(n, 256), 4096), 256, 0, s)(scale, n, 0);
  return launch_status();
}

struct MxArgs {
  const void* x;
  int64_t rows, cols;
  int axis, transpose;
  uint8_t* data;
  uint8_t* scale;
  hipStream_t stream;
};

constexpr int kNotTaken = -1;

// Transposed column cast: the one-read kernel without its row-wise half (16-byte loads, half-wave row split) wherever a lane's kV
// columns are whole; 8192 x 8192 bf16 38.3 vs 40.2 us for mx_col_t_kernel, 16384 x 4096 36.3 vs 41.0 us.
// Wide tiles, more than mx.colt_pipe per CU: a grid of that many workgroups that walk the tiles with the next tile's loads in flight
// (8192 x 8192 bf16 36.4 against 37.5 us, 4096 x 16384 37.1 against 39.2 us; with the row-wise half as well it is slower).
// Tile order: bands of 8 row tiles where the row count allows (8192 x 8192 bf16, wide: 36.6-37.1 us against 38.0-38.6 down the rows
// first), else by shape; narrow tiles, more than 8 per CU: down the rows first (8192 x 8192 38.0 against 38.9, 4096 x 14336 32.4 and 34.4;
// at 4 per CU it loses, 4096 x 4096 11.7 and 10.9).
template <int IN, int OUT, int LAYOUT>
int launch_dual_cols(const MxArgs& a, bool narrow) {
  constexpr int kV = InTraits<IN>::kVec;
  const int64_t bands = ceil_div(a.rows, (int64_t)kDualRows), tiles = bands * ceil_div(a.cols, (int64_t)(32 * kV));
  const int64_t narrow_tiles = bands * dual_col_tiles<16 * kV, LAYOUT>((uint32_t)a.cols), cus = device_facts().cu_count;
  const int64_t pipe_grid = (int64_t)tuning(Knob::mx_colt_pipe) * cus;
  if (tuning(Knob::mx_dual_narrow) >= 0) narrow = tuning(Knob::mx_dual_narrow) != 0;
  if (narrow_tiles > 0x7FFFFFFFll) narrow = false;
  int order = tuning(Knob::mx_dual_order);
  if (order < 0)
    order = narrow && narrow_tiles > 8 * cus ? 0 : a.rows % (8 * kDualRows) == 0 ? 2 : a.cols < a.rows ? 1 : 0;
  if (tiles > 0x7FFFFFFFll) return kNotTaken;
  if (narrow)
    launcher(mx_dual_kernel<IN, OUT, LAYOUT, false, false, 8>, (unsigned)narrow_tiles, kBlock, 0, a.stream)(
        a.x, (uint32_t)a.rows, (uint32_t)a.cols, nullptr, nullptr, a.data, a.scale, order);
  else if constexpr (IN == DT_F32 && OUT == DT_E2M1)
    return kNotTaken;  // mx_col_t_kernel is the better one, see plan_fp4_cols
  else if (pipe_grid > 0 && tiles > pipe_grid)
    launcher(mx_dual_kernel<IN, OUT, LAYOUT, false, true>, (unsigned)pipe_grid, kBlock, 0, a.stream)(
        a.x, (uint32_t)a.rows, (uint32_t)a.cols, nullptr, nullptr, a.data, a.scale, order);
  else
    launcher(mx_dual_kernel<IN, OUT, LAYOUT, false>, (unsigned)tiles, kBlock, 0, a.stream)(
        a.x, (uint32_t)a.rows, (uint32_t)a.cols, nullptr, nullptr, a.data, a.scale, order);
  return launch_status();
}

// Row-wise casts.  Up to 8 MiB of x in passes of one chunk (us, passes of 64 blocks -> of a chunk, blocked scales: bf16 512 x 8192 [8 MiB]
// 3.98 -> 3.83 and 256 x 8192 3.07 -> 2.83, fp32 512 x 4096 4.06 -> 3.64; 16 MiB: bf16 1024 x 8192 6.28 and 6.55, fp32 512 x 8192 5.70
// and 5.85; MXFP4 5.43 and 6.04).  Rows that pad the blocked scales: a workgroup per 256 words, at most one per CU.
constexpr int64_t kSmallRowBytes = (int64_t)8 << 20;
template <int IN, int OUT, int LAYOUT, bool BAND4, bool SMALL>
int launch_rows_as(const MxArgs& a) {
  constexpr int64_t kPass = SMALL ? kWave * InTraits<IN>::kVec / 32 : 64;  // blocks
  const int64_t nblocks = a.rows * a.cols / 32, cus = device_facts().cu_count;
  const int64_t waves = std::min(ceil_div(nblocks, kPass), cus * tuning(Knob::mx_blocks_per_cu) * (kBlock / kWave));
  const int64_t groups = ceil_div(waves, (int64_t)(kBlock / kWave));
  const int64_t pad_words = LAYOUT == DT_SCALE_BLOCKED && a.rows % 128 != 0 ? ceil_div(a.cols, (int64_t)128) * 128 : 0;
  const int64_t pad_groups = std::min(ceil_div(pad_words, (int64_t)kBlock), cus);
  launcher(mx_row_kernel<IN, OUT, LAYOUT, BAND4, SMALL>, (unsigned)(groups + pad_groups), kBlock, 0, a.stream)(
      a.x, (uint32_t)nblocks, (uint32_t)(a.cols / 32), a.data, a.scale, (uint32_t)groups);
  return launch_status();
}
template <int IN, int OUT, int LAYOUT>
int launch_rows(const MxArgs& a) {
  if (a.rows * a.cols * InTraits<IN>::kBytes <= kSmallRowBytes) return launch_rows_as<IN, OUT, LAYOUT, false, true>(a);
  if constexpr (LAYOUT == DT_SCALE_BLOCKED)
    if (a.rows % 128 == 0 && a.cols % 512 == 0 && tuning(Knob::mx_row_band4)) return launch_rows_as<IN, OUT, LAYOUT, true, false>(a);
  return launch_rows_as<IN, OUT, LAYOUT, false, false>(a);
}

template <int IN, int OUT, int LAYOUT>
int launch_mx(const MxArgs& a) {
  constexpr int kV = InTraits<IN>::kVec;
  const int64_t numel = a.rows * a.cols, nblocks = numel / 32;
  const int cus = device_facts().cu_count;
  // x only has to be aligned to its element: the kernels load it through element-aligned vector types
  if (a.axis == 1 && !a.transpose && aligned(a.data, 8) && nblocks < (1ll << 28)) {
    return launch_rows<IN, OUT, LAYOUT>(a);
  }
  if (a.axis == 0 && a.transpose && a.cols % kV == 0 && aligned(a.data, 16) && aligned(a.scale, 4) &&
      a.rows < (1ll << 31) && a.cols < (1ll << 31) && tuning(Knob::mx_colt_via_dual)) {
    const bool narrow = narrow_cols(IN == DT_F32, LAYOUT == DT_SCALE_BLOCKED, a.rows, a.cols, cus);
    const int st = launch_dual_cols<IN, OUT, LAYOUT>(a, narrow);
    if (st != kNotTaken) return st;
  }
  if (a.axis == 0 && a.transpose && a.cols % 4 == 0 && aligned(a.data, 16) && aligned(a.scale, 4) &&
      a.rows < (1ll << 31) && a.cols < (1ll << 31)) {
    const int64_t tiles = ceil_div(a.rows, (int64_t)kColTRows) * ceil_div(a.cols, (int64_t)kColTCols);
    if (tiles <= 0x7FFFFFFFll) {
      launcher(mx_col_t_kernel<IN, OUT, LAYOUT>, (unsigned)tiles, kBlock, 0, a.stream)(a.x, (uint32_t)a.rows, (uint32_t)a.cols,
                                                                              a.data, a.scale);
      return launch_status();
    }
  }
  if (a.axis == 0 && !a.transpose && a.cols % kV == 0 && aligned(a.data, 16) && aligned(a.scale, 8) &&
      a.rows < (1ll << 31) && a.cols < (1ll << 31) && LAYOUT == DT_SCALE_PLAIN) {
    const int64_t tiles = (a.rows / 32) * ceil_div(a.cols, (int64_t)kWave * kV);
    if (tiles <= 0x7FFFFFFFll) {
      int64_t grid = (int64_t)cus * tuning(Knob::mx_col_blocks_per_cu);
      if (grid > tiles) grid = tiles;
      launcher(mx_col_kernel<IN, OUT>, (unsigned)grid, kBlock, 0, a.stream)(a.x, (uint32_t)a.rows, (uint32_t)a.cols, a.data,
                                                                     a.scale, (uint32_t)tiles);
      return launch_status();
    }
  }
  // blocks along the rows with a transposed payload: through the LDS transpose tile
  if constexpr (LAYOUT == DT_SCALE_PLAIN) {
    if (a.axis == 1 && a.transpose && a.rows % 16 == 0 && aligned(a.data, 16) && aligned(a.scale, 4) &&
        a.rows < (1ll << 31) && a.cols < (1ll << 31)) {
      const int64_t tiles = ceil_div(a.rows, (int64_t)kDualRows) * ceil_div(a.cols, (int64_t)(32 * kV));
      if (tiles <= 0x7FFFFFFFll) {
        launcher(mx_row_t_kernel<IN, OUT>, (unsigned)tiles, kBlock, 0, a.stream)(a.x, (uint32_t)a.rows, (uint32_t)a.cols, a.data,
                                                                          a.scale);
        return launch_status();
      }
    }
  }
  // general orientation / alignment
  int64_t outer, inner_blocks, xos, xes, dos, des, s_rows, s_cols;
  int s_t;
  if (a.axis == 1) {
    outer = a.rows; inner_blocks = a.cols / 32; xos = a.cols; xes = 1;
    if (!a.transpose) { dos = a.cols; des = 1; s_rows = a.rows; s_cols = inner_blocks; s_t = 0; }
    else { dos = 1; des = a.rows; s_rows = inner_blocks; s_cols = a.rows; s_t = 1; }
  } else {
    outer = a.cols; inner_blocks = a.rows / 32; xos = 1; xes = a.cols;
    if (!a.transpose) { dos = 1; des = a.cols; s_rows = inner_blocks; s_cols = a.cols; s_t = 1; }
    else { dos = a.rows; des = 1; s_rows = a.cols; s_cols = inner_blocks; s_t = 0; }
  }
  const int64_t total = outer * inner_blocks;
  if (ceil_div(total, kBlock) > 0x7FFFFFFFll) return DT_ERR_INVALID_SHAPE;
  if constexpr (LAYOUT == DT_SCALE_BLOCKED) {
    if (int st = zero_blocked_padding(a.scale, outer, inner_blocks, a.stream)) return st;
  }
  launcher(mx_any_kernel<IN, OUT, LAYOUT>, (unsigned)ceil_div(total, kBlock), kBlock, 0, a.stream)(
      a.x, outer, inner_blocks, xos, xes, dos, des, s_rows, s_cols, s_t, a.data, a.scale);
  return launch_status();
}

template <int IN>
int launch_mx_in(const MxArgs& a, int out_dtype, int layout) {
  if (out_dtype == DT_E4M3FN)
    return layout == DT_SCALE_BLOCKED ? launch_mx<IN, DT_E4M3FN, DT_SCALE_BLOCKED>(a) : launch_mx<IN, DT_E4M3FN, DT_SCALE_PLAIN>(a);
  return layout == DT_SCALE_BLOCKED ? launch_mx<IN, DT_E5M2, DT_SCALE_BLOCKED>(a) : launch_mx<IN, DT_E5M2, DT_SCALE_PLAIN>(a);
}

struct DualArgs {
  const void* x;
  int64_t rows, cols;
  uint8_t *data_r, *scale_r, *data_c, *scale_c;
  hipStream_t stream;
};

// The one-read kernel on `tiles` of 128 rows x 256 (fp32: 128) columns, or, for 16-bit inputs, on tiles half as wide: where the tiles
// are few the narrow ones halve what each lane does and fill the chip (us, wide -> narrow, MXFP8 / MXFP4, bf16: 512 x 512 5.8 -> 4.3 /
// 5.3 -> 4.0, 1024 x 1664 7.2 -> 5.4 / 6.6 -> 5.1, 2048 x 1888 8.3 -> 7.0 / 7.7 -> 6.6, 2752 x 4096, 352 tiles, 11.7 -> 11.0 / 10.3 -> 9.6), and
// where an MXFP8 pair's are four per CU or more and the rows begin on cache lines (8192 x 4096 29.3 -> 27.6, 8192 x 8192 50.7 -> 46.6, 14336 x 4096
// 45.6 -> 42.0, 6240 x 11968 58.6 -> 56.2).  In between, for MXFP4 and for rows off the lines the wide ones win (4096 x 3488, 448 tiles, 14.1
// and 16.5; 6144 x 4096, 768 tiles, 21.5 and 22.3; 8960 x 7520 56.0 and 59.7; MXFP4 8192 x 4096 22.4 and 23.5).
template <int IN, int OUT, int LAYOUT>
int launch_dual_tiles(const DualArgs& a) {
  const int64_t bands = ceil_div(a.rows, (int64_t)kDualRows), tiles = bands * ceil_div(a.cols, (int64_t)32 * InTraits<IN>::kVec);
  const int64_t cus = device_facts().cu_count, narrow_tiles = bands * ceil_div(a.cols, (int64_t)16 * InTraits<IN>::kVec);
  const int knob = tuning(Knob::mx_dual_narrow);
  const bool narrow = IN != DT_F32 && (knob >= 0 ? knob != 0 : tiles * 8 <= cus * 11 || (OUT != DT_E2M1 && tiles >= 4 * cus && a.cols % 64 == 0)) &&
                      narrow_tiles <= 0x7FFFFFFFll;
  const int order = tuning(Knob::mx_dual_order) >= 0 ? tuning(Knob::mx_dual_order) : pair_order(IN == DT_F32, OUT == DT_E2M1, narrow, a.rows, a.cols, cus);
  if constexpr (IN != DT_F32) {
    if (narrow) {
      launcher(mx_dual_kernel<IN, OUT, LAYOUT, true, false, 8>, (unsigned)narrow_tiles, kBlock, 0, a.stream)(
          a.x, (uint32_t)a.rows, (uint32_t)a.cols, a.data_r, a.scale_r, a.data_c, a.scale_c, order);
      return launch_status();
    }
  }
  if (tiles > 0x7FFFFFFFll) return kNotTaken;
  launcher(mx_dual_kernel<IN, OUT, LAYOUT>, (unsigned)tiles, kBlock, 0, a.stream)(a.x, (uint32_t)a.rows, (uint32_t)a.cols, a.data_r,
                                                                           a.scale_r, a.data_c, a.scale_c, order);
  return launch_status();
}

// DT_OK when the one-read kernel was launched, kNotTaken when the shape or an alignment rules it out
template <int IN, int OUT, int LAYOUT>
int launch_dual(const DualArgs& a) {
  if (!aligned(a.data_r, 8) || !aligned(a.data_c, 16) || !aligned(a.scale_r, 4) ||
      !aligned(a.scale_c, 4) || a.rows >= (1ll << 31) || a.cols >= (1ll << 31))
    return kNotTaken;
  return launch_dual_tiles<IN, OUT, LAYOUT>(a);
}
template <int IN>
int launch_dual_in(const DualArgs& a, int out_dtype, int layout) {
  if (out_dtype == DT_E4M3FN)
    return layout == DT_SCALE_BLOCKED ? launch_dual<IN, DT_E4M3FN, DT_SCALE_BLOCKED>(a) : launch_dual<IN, DT_E4M3FN, DT_SCALE_PLAIN>(a);
  return layout == DT_SCALE_BLOCKED ? launch_dual<IN, DT_E5M2, DT_SCALE_BLOCKED>(a) : launch_dual<IN, DT_E5M2, DT_SCALE_PLAIN>(a);
}

}  // namespace

extern "C" int64_t dt_blocked_scale_bytes(int64_t R, int64_t C) {
  if (R < 0 || C < 0) return 0;
  return 128 * dt::ceil_div(R, 128) * 4 * dt::ceil_div(C, 4);
}

extern "C" int dt_mx_fp8_quantize(const void* x, int in_dtype, int64_t rows, int64_t cols, int axis, int transpose,
                                  int out_dtype, int scale_layout, void* data, uint8_t* scale, dt_stream_t stream) {
  if (in_dtype != DT_F32 && in_dtype != DT_BF16 && in_dtype != DT_F16) return DT_ERR_INVALID_DTYPE;
  if (out_dtype != DT_E4M3FN && out_dtype != DT_E5M2) return DT_ERR_INVALID_DTYPE;
  if ((axis != 0 && axis != 1) || (transpose != 0 && transpose != 1)) return DT_ERR_INVALID_MODE;
  if (scale_layout != DT_SCALE_PLAIN && scale_layout != DT_SCALE_BLOCKED) return DT_ERR_INVALID_MODE;
  if (rows < 0 || cols < 0) return DT_ERR_INVALID_SHAPE;
  if ((axis == 1 ? cols : rows) % 32 != 0) return DT_ERR_INVALID_SHAPE;
  // the blocked layout is defined for a scale matrix [outer, inner/32]
  if (scale_layout == DT_SCALE_BLOCKED && !((axis == 1 && !transpose) || (axis == 0 && transpose))) return DT_ERR_INVALID_MODE;
  if (rows == 0 || cols == 0) return DT_OK;
  if (!x || !data || !scale) return DT_ERR_NULL_POINTER;
  if (!dt::aligned(x, in_dtype == DT_F32 ? 4 : 2)) return DT_ERR_MISALIGNED;
  hipStream_t s = dt::as_hip(stream);
  MxArgs a{x, rows, cols, axis, transpose, static_cast<uint8_t*>(data), scale, s};
  switch (in_dtype) {
    case DT_F32: return launch_mx_in<DT_F32>(a, out_dtype, scale_layout);
    case DT_BF16: return launch_mx_in<DT_BF16>(a, out_dtype, scale_layout);
    default: return launch_mx_in<DT_F16>(a, out_dtype, scale_layout);
  }
}

extern "C" int dt_mx_fp8_quantize_dual(const void* x, int in_dtype, int64_t rows, int64_t cols, int out_dtype, int scale_layout,
                                       void* data_rows, uint8_t* scale_rows, void* data_cols_t, uint8_t* scale_cols_t,
                                       dt_stream_t stream) {
  if (in_dtype != DT_F32 && in_dtype != DT_BF16 && in_dtype != DT_F16) return DT_ERR_INVALID_DTYPE;
  if (out_dtype != DT_E4M3FN && out_dtype != DT_E5M2) return DT_ERR_INVALID_DTYPE;
  if (scale_layout != DT_SCALE_PLAIN && scale_layout != DT_SCALE_BLOCKED) return DT_ERR_INVALID_MODE;
  if (rows < 0 || cols < 0 || rows % 32 != 0 || cols % 32 != 0) return DT_ERR_INVALID_SHAPE;
  if (rows == 0 || cols == 0) return DT_OK;
  if (!x || !data_rows || !scale_rows || !data_cols_t || !scale_cols_t) return DT_ERR_NULL_POINTER;
  if (!dt::aligned(x, in_dtype == DT_F32 ? 4 : 2)) return DT_ERR_MISALIGNED;
  hipStream_t s = dt::as_hip(stream);
  DualArgs a{x, rows, cols, static_cast<uint8_t*>(data_rows), scale_rows, static_cast<uint8_t*>(data_cols_t), scale_cols_t, s};
  const bool fast_ok = dt::tuning(dt::Knob::mx_dual) != 0;
  if (fast_ok) {
    int st;
    switch (in_dtype) {
      case DT_F32: st = launch_dual_in<DT_F32>(a, out_dtype, scale_layout); break;
      case DT_BF16: st = launch_dual_in<DT_BF16>(a, out_dtype, scale_layout); break;
      default: st = launch_dual_in<DT_F16>(a, out_dtype, scale_layout); break;
    }
    if (st != kNotTaken) return st;
  }
  // two passes over x
  if (int st = dt_mx_fp8_quantize(x, in_dtype, rows, cols, 1, 0, out_dtype, scale_layout, data_rows, scale_rows, stream)) return st;
  return dt_mx_fp8_quantize(x, in_dtype, rows, cols, 0, 1, out_dtype, scale_layout, data_cols_t, scale_cols_t, stream);
}

namespace {
// blocks down the columns, payload transposed: [cols, rows/2], scales [cols, rows/32]
template <int IN, int LAYOUT>
int launch_mx_fp4_cols(const MxArgs& a) {
  // As for MXFP8, the one-read kernel without its row-wise half, where plan_fp4_cols prefers it
  constexpr int kV = InTraits<IN>::kVec;
  const int64_t cus = device_facts().cu_count;
  const Fp4Cols plan = plan_fp4_cols(IN == DT_F32, LAYOUT == DT_SCALE_BLOCKED, a.rows, a.cols, cus, (int64_t)tuning(Knob::mx_colt_pipe) * cus,
                                     tuning(Knob::mx_dual_narrow));
  if (a.cols % kV == 0 && tuning(Knob::mx_colt_via_dual) && plan != kFp4ColT) {
    const int st = launch_dual_cols<IN, DT_E2M1, LAYOUT>(a, plan == kFp4Narrow);
    if (st != kNotTaken) return st;
  }
  const int64_t tiles = ceil_div(a.rows, (int64_t)kColTRows) * ceil_div(a.cols, (int64_t)kColTCols);
  if (tiles > 0x7FFFFFFFll) return DT_ERR_INVALID_SHAPE;
  launcher(mx_col_t_kernel<IN, DT_E2M1, LAYOUT>, (unsigned)tiles, kBlock, 0, a.stream)(a.x, (uint32_t)a.rows, (uint32_t)a.cols, a.data,
                                                                                a.scale);
  return launch_status();
}
}  // namespace

extern "C" int dt_mx_fp4_quantize(const void* x, int in_dtype, int64_t rows, int64_t cols, int axis, int scale_layout,
                                  void* data, uint8_t* scale, dt_stream_t stream) {
  if (in_dtype != DT_F32 && in_dtype != DT_BF16 && in_dtype != DT_F16) return DT_ERR_INVALID_DTYPE;
  if (axis != 0 && axis != 1) return DT_ERR_INVALID_MODE;
  if (scale_layout != DT_SCALE_PLAIN && scale_layout != DT_SCALE_BLOCKED) return DT_ERR_INVALID_MODE;
  if (rows < 0 || cols < 0 || (axis == 1 ? cols : rows) % 32 != 0) return DT_ERR_INVALID_SHAPE;
  if (rows == 0 || cols == 0) return DT_OK;
  if (!x || !data || !scale) return DT_ERR_NULL_POINTER;
  hipStream_t s = dt::as_hip(stream);
  const bool blocked = scale_layout == DT_SCALE_BLOCKED;
  if (axis == 0) {
    // a lane loads 4 adjacent columns of a row with one 8- or 16-byte load
    const int64_t kB = in_dtype == DT_F32 ? 4 : 2;
    if (cols % 4 != 0 || rows >= (1ll << 31) || cols >= (1ll << 31)) return DT_ERR_INVALID_SHAPE;
    if (!dt::aligned(x, 4 * kB) || (cols * kB) % (4 * kB) != 0 || !dt::aligned(data, 16) || !dt::aligned(scale, 4))
      return DT_ERR_MISALIGNED;
    MxArgs a{x, rows, cols, 0, 1, static_cast<uint8_t*>(data), scale, s};
    switch (in_dtype) {
      case DT_F32: return blocked ? launch_mx_fp4_cols<DT_F32, DT_SCALE_BLOCKED>(a) : launch_mx_fp4_cols<DT_F32, DT_SCALE_PLAIN>(a);
      case DT_BF16: return blocked ? launch_mx_fp4_cols<DT_BF16, DT_SCALE_BLOCKED>(a) : launch_mx_fp4_cols<DT_BF16, DT_SCALE_PLAIN>(a);
      default: return blocked ? launch_mx_fp4_cols<DT_F16, DT_SCALE_BLOCKED>(a) : launch_mx_fp4_cols<DT_F16, DT_SCALE_PLAIN>(a);
    }
  }
  if (rows * cols / 32 >= (1ll << 28)) return DT_ERR_INVALID_SHAPE;  // block indices are 32 bits wide in the kernel
  if (!dt::aligned(x, 16) || !dt::aligned(data, 4)) return DT_ERR_MISALIGNED;
  MxArgs a{x, rows, cols, 1, 0, static_cast<uint8_t*>(data), scale, s};
  switch (in_dtype) {
    case DT_F32: return blocked ? launch_rows<DT_F32, DT_E2M1, DT_SCALE_BLOCKED>(a) : launch_rows<DT_F32, DT_E2M1, DT_SCALE_PLAIN>(a);
    case DT_BF16: return blocked ? launch_rows<DT_BF16, DT_E2M1, DT_SCALE_BLOCKED>(a) : launch_rows<DT_BF16, DT_E2M1, DT_SCALE_PLAIN>(a);
    default: return blocked ? launch_rows<DT_F16, DT_E2M1, DT_SCALE_BLOCKED>(a) : launch_rows<DT_F16, DT_E2M1, DT_SCALE_PLAIN>(a);
  }
}

namespace {
// both MXFP4 operands of one tensor from a single read: mx_dual_kernel with the e2m1 output code
template <int IN, int LAYOUT>
int launch_dual_fp4(const DualArgs& a) {
  if (!aligned(a.data_r, 4) || !aligned(a.data_c, 16) || !aligned(a.scale_r, 4) || !aligned(a.scale_c, 4) ||
      a.rows >= (1ll << 31) || a.cols >= (1ll << 31))
    return kNotTaken;
  return launch_dual_tiles<IN, DT_E2M1, LAYOUT>(a);
}
template <int IN>
int launch_dual_fp4_in(const DualArgs& a, int layout) {
  return layout == DT_SCALE_BLOCKED ? launch_dual_fp4<IN, DT_SCALE_BLOCKED>(a) : launch_dual_fp4<IN, DT_SCALE_PLAIN>(a);
}
}  // namespace

extern "C" int dt_mx_fp4_quantize_dual(const void* x, int in_dtype, int64_t rows, int64_t cols, int scale_layout, void* data_rows,
                                       uint8_t* scale_rows, void* data_cols_t, uint8_t* scale_cols_t, dt_stream_t stream) {
  if (in_dtype != DT_F32 && in_dtype != DT_BF16 && in_dtype != DT_F16) return DT_ERR_INVALID_DTYPE;
  if (scale_layout != DT_SCALE_PLAIN && scale_layout != DT_SCALE_BLOCKED) return DT_ERR_INVALID_MODE;
  if (rows < 0 || cols < 0 || rows % 32 != 0 || cols % 32 != 0) return DT_ERR_INVALID_SHAPE;
  if (rows == 0 || cols == 0) return DT_OK;
  if (!x || !data_rows || !scale_rows || !data_cols_t || !scale_cols_t) return DT_ERR_NULL_POINTER;
  if (!dt::aligned(x, in_dtype == DT_F32 ? 4 : 2)) return DT_ERR_MISALIGNED;
  hipStream_t s = dt::as_hip(stream);
  DualArgs a{x, rows, cols, static_cast<uint8_t*>(data_rows), scale_rows, static_cast<uint8_t*>(data_cols_t), scale_cols_t, s};
  if (dt::tuning(dt::Knob::mx_dual) != 0) {
    int st;
    switch (in_dtype) {
      case DT_F32: st = launch_dual_fp4_in<DT_F32>(a, scale_layout); break;
      case DT_BF16: st = launch_dual_fp4_in<DT_BF16>(a, scale_layout); break;
      default: st = launch_dual_fp4_in<DT_F16>(a, scale_layout); break;
    }
    if (st != kNotTaken) return st;
  }
  // two passes over x
  if (int st = dt_mx_fp4_quantize(x, in_dtype, rows, cols, 1, scale_layout, data_rows, scale_rows, stream)) return st;
  return dt_mx_fp4_quantize(x, in_dtype, rows, cols, 0, scale_layout, data_cols_t, scale_cols_t, stream);
}

extern "C" int dt_to_blocked(const uint8_t* scale, int64_t R, int64_t C, uint8_t* out, dt_stream_t stream) {
  if (R < 0 || C < 0) return DT_ERR_INVALID_SHAPE;
  if (R == 0 || C == 0) return DT_OK;
  if (!scale || !out) return DT_ERR_NULL_POINTER;
  hipStream_t s = dt::as_hip(stream);
  const int64_t groups = dt_blocked_scale_bytes(R, C) / 16;
  if (dt::ceil_div(R * C, 256) > 0x7FFFFFFFll) return DT_ERR_INVALID_SHAPE;
  const unsigned grid = (unsigned)std::min<int64_t>(dt::ceil_div(groups, (int64_t)dt::kBlock), (int64_t)dt::device_facts().cu_count * 16);
  if (R * C < 4) dt::launcher(dt::to_blocked_kernel<true, uint32_t>, grid, dt::kBlock, 0, s)(scale, R, C, groups, out);
  else if ((groups >> 5) <= 0xFFFFFFFFll) dt::launcher(dt::to_blocked_kernel<false, uint32_t>, grid, dt::kBlock, 0, s)(scale, R, C, groups, out);
  else dt::launcher(dt::to_blocked_kernel<false, uint64_t>, grid, dt::kBlock, 0, s)(scale, R, C, groups, out);
  return dt::launch_status();
}
