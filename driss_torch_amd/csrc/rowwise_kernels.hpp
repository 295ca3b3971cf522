// Row-wise dynamic quantization: per-row amax -> scale -> saturating fp8 cast.
//
// Fast path: one wavefront owns one row and keeps it in registers between the reduction
// and the cast, so the row is read from memory once; no LDS and no barrier is involved.
// Longer rows take a workgroup each and stay in its registers the same way; only rows longer than 16384
// vectors are read twice.  Rows of any width keep these kernels (RowSpan).
#pragma once

#include "quant_kernels.hpp"

namespace dt {

constexpr int kRowsPerBlock = kBlock / kWave;  // one wave per row

// A row of a matrix whose width is no whole number of vectors (EDGES; base aligned to a vector, output to its
// packed store): element f of the flat tensor sits in vector f / kV of x and of the output whatever row it
// belongs to, so a row is `head` elements up to the first vector boundary, whole aligned vectors, and `tail`
// elements.  Lanes 0 .. head - 1 and kV .. kV + tail - 1 of the row's first wave take one of those elements each.
// (Before, every access of such a row was a vector at the row's own alignment, which costs the second line of
// each straddled one, and loads went without the streaming hint: 8192 x 8190 bf16 37.5 -> 33.9 us; rows of up
// to 256 vectors had a workgroup of four waves each as well.)
template <int IN, bool EDGES>
struct RowSpan {
  static constexpr int kV = InTraits<IN>::kVec;
  int64_t vec0;       // first whole vector
  int nvec;           // whole vectors
  int64_t edge = -1;  // this lane's single element, flat; -1: none
  __device__ RowSpan(int64_t row, int64_t cols, int lane_of_row) {
    const int64_t first = row * cols;
    if constexpr (EDGES) {
      const int head = (int)(-first & (kV - 1));
      vec0 = (first + head) / kV;
      nvec = (int)((cols - head) / kV);
      const int tail = (int)(cols - head) - nvec * kV;
      if (lane_of_row < head) edge = first + lane_of_row;
      else if (lane_of_row >= kV && lane_of_row < kV + tail) edge = (vec0 + nvec) * kV + lane_of_row - kV;
    } else {
      vec0 = first / kV;
      nvec = (int)(cols / kV);
    }
  }
};

template <int IN, int OUT, int NV, bool EDGES = false>
__global__ __launch_bounds__(kBlock) void rowwise_wave_kernel(const void* __restrict__ x, int64_t rows,
                                                              int64_t cols, uint8_t* __restrict__ out,
                                                              float* __restrict__ amax_out,
                                                              float* __restrict__ scale_out) {
  saturate_fp8_conversions();
  const int lane = threadIdx.x % kWave;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + threadIdx.x / kWave;
  if (row >= rows) return;  // whole wave leaves together; the kernel has no barrier
  const RowSpan<IN, EDGES> span(row, cols, lane);
  const int row_vecs = span.nvec;
  const u32x4* v = static_cast<const u32x4*>(x) + span.vec0;
  u32x4 w[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = lane + u * kWave;
    w[u] = j < row_vecs ? ld_stream(v + j) : u32x4{0u, 0u, 0u, 0u};
  }
  uint32_t e = 0;  // the lane's single element as fp32 bits
  if (EDGES && span.edge >= 0) e = fp32_bits_of<IN>(x, span.edge);
  uint32_t m = 0;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if constexpr (IN == DT_F32) {
      m = umax(m, umax(umax(absbits_f32(w[u].x), absbits_f32(w[u].y)), umax(absbits_f32(w[u].z), absbits_f32(w[u].w))));
    } else {
      m = pk_absmax16(pk_absmax16(m, w[u].x), w[u].y);
      m = pk_absmax16(pk_absmax16(m, w[u].z), w[u].w);
    }
  }
  if constexpr (IN != DT_F32) m = umax(m & 0xFFFFu, m >> 16) << 16;
  if constexpr (EDGES) m = umax(m, absbits_f32(e));
  m = wave_umax(m);
  const float amax = as_f32(m);
  const float s = amax_to_scale(amax, fp8_max<OUT>());
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = lane + u * kWave;
    if (j < row_vecs) cast_vec<IN, OUT, false>(w[u], s, out, span.vec0 + j);
  }
  if (EDGES && span.edge >= 0) out[span.edge] = (uint8_t)pack4<OUT>(scaled<false>(as_f32(e), s), 0.f, 0.f, 0.f);
  if (lane == 0) {
    if (amax_out) amax_out[row] = amax;
    if (scale_out) scale_out[row] = s;
  }
}

// Longer rows: one workgroup per row, NV vectors per lane kept in registers between the reduction
// (one LDS exchange between the four waves) and the cast: still a single read of the row.
// kRowsEdges: rows of any width on an aligned base (RowSpan).  kRowsAny: x or the output not aligned for
// that (cols % kV = tail elements, done by the first lanes): the same loads and stores through vector types
// that claim only element / byte alignment, as in cast_kernel_unaligned.
enum RowAccess { kRowsWhole = 0, kRowsEdges = 1, kRowsAny = 2 };
template <int IN, int OUT, int NV, int ACCESS = kRowsWhole>
__global__ __launch_bounds__(kBlock) void rowwise_block_resident_kernel(const void* __restrict__ x, int64_t cols,
                                                                        uint8_t* __restrict__ out,
                                                                        float* __restrict__ amax_out,
                                                                        float* __restrict__ scale_out) {
  constexpr int kV = InTraits<IN>::kVec, kB = InTraits<IN>::kBytes;
  constexpr bool ANY = ACCESS == kRowsAny, EDGES = ACCESS == kRowsEdges;
  saturate_fp8_conversions();
  __shared__ uint32_t lds[kBlock / kWave];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const RowSpan<IN, EDGES> span(row, cols, tid);
  const int row_vecs = span.nvec, tail = ANY ? (int)(cols % kV) : 0;
  const uint8_t* xrow = static_cast<const uint8_t*>(x) + row * cols * kB;  // ANY
  const u32x4* v = static_cast<const u32x4*>(x) + span.vec0;
  u32x4 w[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = tid + u * kBlock;
    if constexpr (ANY) {
      typedef typename std::conditional<IN == DT_F32, u32x4_elem4, u32x4_elem2>::type vec_t;
      w[u] = j < row_vecs ? reinterpret_cast<const vec_t*>(xrow)[j] : u32x4{0u, 0u, 0u, 0u};
    } else {
      w[u] = j < row_vecs ? ld_stream(v + j) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  uint32_t e = 0;  // the lane's single element as fp32 bits
  if (EDGES && span.edge >= 0) e = fp32_bits_of<IN>(x, span.edge);
  uint32_t m = 0;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if constexpr (IN == DT_F32) {
      m = umax(m, umax(umax(absbits_f32(w[u].x), absbits_f32(w[u].y)), umax(absbits_f32(w[u].z), absbits_f32(w[u].w))));
    } else {
      m = pk_absmax16(pk_absmax16(m, w[u].x), w[u].y);
      m = pk_absmax16(pk_absmax16(m, w[u].z), w[u].w);
    }
  }
  if constexpr (IN != DT_F32) m = umax(m & 0xFFFFu, m >> 16) << 16;
  if constexpr (EDGES) m = umax(m, absbits_f32(e));
  if constexpr (ANY) {
    if (tid < tail) m = umax(m, absbits_of<IN>(xrow, (int64_t)row_vecs * kV + tid));
  }
  m = block_umax<kBlock / kWave>(m, lds);
  const float amax = as_f32(m);
  const float s = amax_to_scale(amax, fp8_max<OUT>());
  uint8_t* orow = out + row * cols;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = tid + u * kBlock;
    if (j < row_vecs) {
      if constexpr (ANY) {
        uint32_t r[kV / 4];
        cast_vec_to_words<IN, OUT, false>(w[u], s, r);
        if constexpr (IN == DT_F32) *reinterpret_cast<u32_byte*>(orow + (int64_t)j * 4) = r[0];
        else *reinterpret_cast<u32x2_byte*>(orow + (int64_t)j * 8) = u32x2{r[0], r[1]};
      } else {
        cast_vec<IN, OUT, false>(w[u], s, out, span.vec0 + j);
      }
    }
  }
  if (EDGES && span.edge >= 0) out[span.edge] = (uint8_t)pack4<OUT>(scaled<false>(as_f32(e), s), 0.f, 0.f, 0.f);
  if constexpr (ANY) {
    if (tid < tail) orow[(int64_t)row_vecs * kV + tid] = cast_one<IN, OUT, false>(xrow, (int64_t)row_vecs * kV + tid, s);
  }
  if (tid == 0) {
    if (amax_out) amax_out[row] = amax;
    if (scale_out) scale_out[row] = s;
  }
}

// One workgroup per row; VEC selects 16-byte access (aligned rows) or element access.
template <int IN, int OUT, bool VEC>
__global__ __launch_bounds__(kBlock) void rowwise_block_kernel(const void* __restrict__ x, int64_t cols,
                                                               uint8_t* __restrict__ out,
                                                               float* __restrict__ amax_out,
                                                               float* __restrict__ scale_out) {
  constexpr int kB = InTraits<IN>::kBytes, kV = InTraits<IN>::kVec;
  saturate_fp8_conversions();
  __shared__ uint32_t lds[kBlock / kWave];
  const int64_t row = blockIdx.x;
  const uint8_t* xrow = static_cast<const uint8_t*>(x) + row * cols * kB;
  uint8_t* orow = out + row * cols;
  const int tid = threadIdx.x;
  uint32_t m = 0;
  if constexpr (VEC) {
    const u32x4* v = reinterpret_cast<const u32x4*>(xrow);
    for (int64_t j = tid; j < cols / kV; j += kBlock) {
      u32x4 w = v[j];
      if constexpr (IN == DT_F32) {
        m = umax(m, umax(umax(absbits_f32(w.x), absbits_f32(w.y)), umax(absbits_f32(w.z), absbits_f32(w.w))));
      } else {
        uint32_t p = pk_absmax16(pk_absmax16(pk_absmax16(pk_absmax16(0u, w.x), w.y), w.z), w.w);
        m = umax(m, umax(p & 0xFFFFu, p >> 16) << 16);
      }
    }
  } else {
    for (int64_t j = tid; j < cols; j += kBlock) m = umax(m, absbits_of<IN>(xrow, j));
  }
  m = block_umax<kBlock / kWave>(m, lds);
  const float amax = as_f32(m);
  const float s = amax_to_scale(amax, fp8_max<OUT>());
  if constexpr (VEC) {
    const u32x4* v = reinterpret_cast<const u32x4*>(xrow);
    for (int64_t j = tid; j < cols / kV; j += kBlock) cast_vec<IN, OUT, false>(v[j], s, orow, j);
  } else {
    for (int64_t j = tid; j < cols; j += kBlock) orow[j] = cast_one<IN, OUT, false>(xrow, j, s);
  }
  if (tid == 0) {
    if (amax_out) amax_out[row] = amax;
    if (scale_out) scale_out[row] = s;
  }
}

template <int IN, int OUT>
inline int launch_rowwise_impl(const void* x, int64_t rows, int64_t cols, void* out, float* amax_out,
                               float* scale_out, hipStream_t stream) {
  constexpr int kV = InTraits<IN>::kVec;
  constexpr size_t kStoreAlign = IN == DT_F32 ? 4 : 8;
  uint8_t* o = static_cast<uint8_t*>(out);
  const bool base_ok = aligned(x, 16) && aligned(out, kStoreAlign), vec_ok = base_ok && cols % kV == 0;
  const int64_t row_vecs = cols / kV;
  const int64_t block_from = tuning("rowwise.block_from_vecs");  // rows at least this long take a workgroup each
  const bool held = row_vecs >= 1 && row_vecs <= 64 * kBlock && rows <= 0x7FFFFFFFll;  // a workgroup can hold a row
#define DT_ROWB(NV, ACCESS) \
  rowwise_block_resident_kernel<IN, OUT, NV, ACCESS><<<(unsigned)rows, kBlock, 0, stream>>>(x, cols, o, amax_out, scale_out)
#define DT_ROWB_ANY_LENGTH(ACCESS)                     \
  do {                                                 \
    if (row_vecs <= 1 * kBlock) DT_ROWB(1, ACCESS);    \
    else if (row_vecs <= 2 * kBlock) DT_ROWB(2, ACCESS);   \
    else if (row_vecs <= 4 * kBlock) DT_ROWB(4, ACCESS);   \
    else if (row_vecs <= 8 * kBlock) DT_ROWB(8, ACCESS);   \
    else if (row_vecs <= 16 * kBlock) DT_ROWB(16, ACCESS); \
    else if (row_vecs <= 32 * kBlock) DT_ROWB(32, ACCESS); \
    else DT_ROWB(64, ACCESS);                          \
  } while (0)
  const unsigned wave_grid = (unsigned)ceil_div(rows, kRowsPerBlock);
#define DT_ROW(NV, EDGES) rowwise_wave_kernel<IN, OUT, NV, EDGES><<<wave_grid, kBlock, 0, stream>>>(x, rows, cols, o, amax_out, scale_out)
#define DT_ROW_ANY_LENGTH(EDGES)                      \
  do {                                                \
    if (row_vecs <= 1 * kWave) DT_ROW(1, EDGES);      \
    else if (row_vecs <= 2 * kWave) DT_ROW(2, EDGES); \
    else if (row_vecs <= 4 * kWave) DT_ROW(4, EDGES); \
    else if (row_vecs <= 8 * kWave) DT_ROW(8, EDGES); \
    else DT_ROW(16, EDGES);                           \
  } while (0)
  if (vec_ok && row_vecs >= block_from && held) {
    DT_ROWB_ANY_LENGTH(kRowsWhole);
  } else if (base_ok && !vec_ok && held) {  // rows that are not whole vectors, on an aligned base
    if (row_vecs >= block_from || row_vecs > 16 * kWave) DT_ROWB_ANY_LENGTH(kRowsEdges);
    else DT_ROW_ANY_LENGTH(true);
  } else if (!vec_ok && held) {  // x or the output not aligned: a workgroup per row with element-aligned vector accesses
    DT_ROWB_ANY_LENGTH(kRowsAny);
  } else if (vec_ok && row_vecs <= 16 * kWave) {
    DT_ROW_ANY_LENGTH(false);
#undef DT_ROWB
#undef DT_ROWB_ANY_LENGTH
#undef DT_ROW
#undef DT_ROW_ANY_LENGTH
  } else if (vec_ok) {
    rowwise_block_kernel<IN, OUT, true><<<(unsigned)rows, kBlock, 0, stream>>>(x, cols, o, amax_out, scale_out);
  } else {
    rowwise_block_kernel<IN, OUT, false><<<(unsigned)rows, kBlock, 0, stream>>>(x, cols, o, amax_out, scale_out);
  }
  return launch_status();
}

inline int launch_rowwise(const void* x, int in_dtype, int64_t rows, int64_t cols, int out_dtype, void* out,
                          float* amax_out, float* scale_out, hipStream_t stream) {
  if (rows > 0x7FFFFFFFll) return DT_ERR_INVALID_SHAPE;
  if (in_dtype == DT_F32) {
    if (out_dtype == DT_E4M3FN) return launch_rowwise_impl<DT_F32, DT_E4M3FN>(x, rows, cols, out, amax_out, scale_out, stream);
    return launch_rowwise_impl<DT_F32, DT_E5M2>(x, rows, cols, out, amax_out, scale_out, stream);
  }
  if (out_dtype == DT_E4M3FN) return launch_rowwise_impl<DT_BF16, DT_E4M3FN>(x, rows, cols, out, amax_out, scale_out, stream);
  return launch_rowwise_impl<DT_BF16, DT_E5M2>(x, rows, cols, out, amax_out, scale_out, stream);
}

}  // namespace dt
