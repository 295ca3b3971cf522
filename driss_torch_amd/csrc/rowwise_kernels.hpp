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

// A row of a matrix on an aligned base (x aligned to a vector, the output to its packed store).  Where the width
// is no whole number of vectors (EDGES), element f of the flat tensor still sits in vector f / kV of x and of the
// output whatever row it belongs to, so a row is `head` elements up to the first vector boundary, whole aligned
// vectors, and `tail` elements.  Lanes 0 .. head - 1 and kV .. kV + tail - 1 of the row's first wave take one of
// those elements each.  (Before, every access of such a row was a vector at the row's own alignment, which costs
// the second line of each straddled one, and loads went without the streaming hint: 8192 x 8190 bf16 37.5 ->
// 33.9 us; rows of up to 256 vectors had a workgroup of four waves each as well.)
//
// The row is read through a buffer descriptor whose length ends it: a load past its end returns zeros and asks
// memory nothing, so no load stands under a test.  (Under tests, each with zeros to merge when it fails, the
// compiler may put a wait and a copy behind a load, one memory latency more per row: us, fp32 1000 x 1000 3.65 -> 3.17,
// bf16 2071 x 1952 4.5 -> 4.2.)
template <int IN, bool EDGES>
struct RowSpan {
  static constexpr int kV = InTraits<IN>::kVec, kB = InTraits<IN>::kBytes;
  int64_t from;    // the vector that the row's first element lies in
  int64_t vec0;    // first whole vector
  int nvec;        // whole vectors
  int skip, tail;  // elements of vector `from` that are the row's before; elements behind the last whole vector
  __amdgpu_buffer_rsrc_t vectors;
  // row, cols: the same for the whole wave
  __device__ RowSpan(const void* x, int64_t row, int64_t cols) {
    const uint64_t first = (uint64_t)row * (uint64_t)cols;
    from = (int64_t)(first / kV);
    skip = EDGES ? (int)(first % kV) : 0;
    vec0 = from + (skip != 0);
    const int64_t rest = cols - (skip ? kV - skip : 0);
    nvec = (int)((uint64_t)rest / kV);
    tail = EDGES ? (int)((uint64_t)rest % kV) : 0;
    vectors = descriptor(x, vec0, nvec * 16);
  }
  __device__ u32x4 load(int j) const {  // vector j of the row, or zeros
    return __builtin_amdgcn_raw_buffer_load_b128(vectors, j * 16, 0, kStreaming);
  }
  __device__ int edge(int lane_of_row) const {  // the lane's single element, counted from vector `from`; -1: none
    const int head = skip ? kV - skip : 0;
    const int at_tail = (int)(vec0 - from + nvec - 1) * kV + lane_of_row;
    return lane_of_row < head ? skip + lane_of_row : lane_of_row >= kV && lane_of_row < kV + tail ? at_tail : -1;
  }
  __device__ uint32_t load_edge(const void* x, int64_t cols, int edge) const {  // that element as fp32 bits, or zero
    const __amdgpu_buffer_rsrc_t elements = descriptor(x, from, (skip + (int)cols) * kB);
    const int at = edge >= 0 ? edge * kB : 1 << 30;  // past the end of any row
    if constexpr (IN == DT_F32) return __builtin_amdgcn_raw_buffer_load_b32(elements, at, 0, 0);
    else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(elements, at, 0, 0) << 16;
  }

 private:
  static constexpr int kStreaming = 2;  // the nt bit
  __device__ static __amdgpu_buffer_rsrc_t descriptor(const void* x, int64_t vec, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(static_cast<const u32x4*>(x) + vec), 0, bytes, 0x00027000);
  }
};

// kRowsWhole: rows of whole vectors on an aligned base.  kRowsEdges: of any width, there (RowSpan).  kRowsAny: x or
// the output not aligned for that (cols % kV = tail elements, done by the first lanes): loads and stores through
// vector types that claim only element / byte alignment, as in cast_kernel_unaligned.
// kRowsEdgesCached: kRowsEdges with plain stores.  Rows between vectors share lines of the output, and so do the waves
// of a row; a streaming store sends its part of such a line alone, which pays once the output does not stay in the
// caches anyway (us, streaming and plain, bf16: 100 x 1001 2.74 and 2.47; into an output that was written shortly
// before, 2000 x 1001 3.84 and 3.41, 512 x 5121 4.17 and 4.00, 8192 x 8190 34.7 and 34.4; into outputs that are
// kept, 3.85 and 3.99, 4.28 and 4.71, 34.8 and 37.4).
enum RowAccess { kRowsWhole = 0, kRowsEdges = 1, kRowsAny = 2, kRowsEdgesCached = 3 };
constexpr int64_t kStreamEdgesFrom = (int64_t)2 << 20;  // bytes of output

template <int IN, int OUT, int ACCESS>
__device__ __forceinline__ void cast_row_vec(u32x4 w, float s, uint8_t* __restrict__ out, int j) {
  if constexpr (ACCESS != kRowsEdgesCached) {
    cast_vec<IN, OUT, false>(w, s, out, j);
  } else {
    uint32_t r[InTraits<IN>::kVec / 4];
    cast_vec_to_words<IN, OUT, false>(w, s, r);
    if constexpr (IN == DT_F32) reinterpret_cast<uint32_t*>(out)[j] = r[0];
    else reinterpret_cast<u32x2*>(out)[j] = u32x2{r[0], r[1]};
  }
}

template <int IN, int OUT, int NV, int ACCESS = kRowsWhole>
__global__ __launch_bounds__(kBlock) void rowwise_wave_kernel(const void* __restrict__ x, int64_t rows,
                                                              int64_t cols, uint8_t* __restrict__ out,
                                                              float* __restrict__ amax_out,
                                                              float* __restrict__ scale_out) {
  constexpr bool EDGES = ACCESS != kRowsWhole;
  saturate_fp8_conversions();
  const int lane = threadIdx.x % kWave;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (row >= rows) return;  // whole wave leaves together; the kernel has no barrier
  const RowSpan<IN, EDGES> span(x, row, cols);
  const int row_vecs = span.nvec;
  u32x4 w[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) w[u] = span.load(lane + u * kWave);
  const int edge = EDGES ? span.edge(lane) : -1;
  const uint32_t e = EDGES ? span.load_edge(x, cols, edge) : 0u;  // the lane's single element as fp32 bits
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
  uint8_t* const ovec = out + span.vec0 * InTraits<IN>::kVec;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = lane + u * kWave;
    if (j < row_vecs) cast_row_vec<IN, OUT, ACCESS>(w[u], s, ovec, j);
  }
  if (EDGES && edge >= 0) out[span.from * InTraits<IN>::kVec + edge] = (uint8_t)pack4<OUT>(scaled<false>(as_f32(e), s), 0.f, 0.f, 0.f);
  if (lane == 0) {
    if (amax_out) amax_out[row] = amax;
    if (scale_out) scale_out[row] = s;
  }
}

// Longer rows: one workgroup per row, NV vectors per lane kept in registers between the reduction
// (one LDS exchange between the four waves) and the cast: still a single read of the row.
template <int IN, int OUT, int NV, int ACCESS = kRowsWhole>
__global__ __launch_bounds__(kBlock) void rowwise_block_resident_kernel(const void* __restrict__ x, int64_t cols,
                                                                        uint8_t* __restrict__ out,
                                                                        float* __restrict__ amax_out,
                                                                        float* __restrict__ scale_out) {
  constexpr int kV = InTraits<IN>::kVec, kB = InTraits<IN>::kBytes;
  constexpr bool ANY = ACCESS == kRowsAny, EDGES = ACCESS == kRowsEdges || ACCESS == kRowsEdgesCached;
  saturate_fp8_conversions();
  __shared__ uint32_t lds[kBlock / kWave];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const RowSpan<IN, EDGES> span(x, row, cols);
  const int row_vecs = span.nvec, tail = ANY ? (int)(cols % kV) : 0;
  const uint8_t* xrow = static_cast<const uint8_t*>(x) + row * cols * kB;  // ANY
  const u32x4* v = static_cast<const u32x4*>(x) + span.vec0;
  int edge = -1;
  uint32_t e = 0;  // the lane's single element as fp32 bits
  auto load_edge = [&]() {
    edge = span.edge(tid);
    e = span.load_edge(x, cols, edge);
  };
  if constexpr (EDGES && NV > 8) load_edge();  // (behind loads under a test it would be asked for when they have all arrived)
  u32x4 w[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int j = tid + u * kBlock;
    if constexpr (ANY) {
      typedef typename std::conditional<IN == DT_F32, u32x4_elem4, u32x4_elem2>::type vec_t;
      w[u] = j < row_vecs ? reinterpret_cast<const vec_t*>(xrow)[j] : u32x4{0u, 0u, 0u, 0u};
    } else if constexpr (NV <= 8) {
      w[u] = span.load(j);
    } else {  // (up to half of the loads would ask for nothing, which costs their issue: 1000 x 20000 fp32 19.2 -> 19.8 us)
      w[u] = j < row_vecs ? ld_stream(v + j) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  if constexpr (EDGES && NV <= 8) load_edge();
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
  uint8_t* orow = out + row * cols;  // ANY
  uint8_t* const ovec = out + span.vec0 * kV;
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
        cast_row_vec<IN, OUT, ACCESS>(w[u], s, ovec, j);
      }
    }
  }
  if (EDGES && edge >= 0) out[span.from * kV + edge] = (uint8_t)pack4<OUT>(scaled<false>(as_f32(e), s), 0.f, 0.f, 0.f);
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
  const int64_t block_from = tuning(Knob::rowwise_block_from_vecs);  // rows at least this long take a workgroup each
  const bool held = row_vecs >= 1 && row_vecs <= 64 * kBlock && rows <= 0x7FFFFFFFll;  // a workgroup can hold a row
  const bool edges_cached = rows * cols < kStreamEdgesFrom;
#define DT_ROWB(NV, ACCESS) \
  launcher(rowwise_block_resident_kernel<IN, OUT, NV, ACCESS>, (unsigned)rows, kBlock, 0, stream)(x, cols, o, amax_out, scale_out)
#define DT_ROWB_ANY_LENGTH(ACCESS, SHORT_ACCESS)       \
  do {                                                 \
    if (row_vecs <= 1 * kBlock) DT_ROWB(1, SHORT_ACCESS);    \
    else if (row_vecs <= 2 * kBlock) DT_ROWB(2, SHORT_ACCESS);   \
    else if (row_vecs <= 4 * kBlock) DT_ROWB(4, SHORT_ACCESS);   \
    else if (row_vecs <= 8 * kBlock) DT_ROWB(8, SHORT_ACCESS);   \
    else if (row_vecs <= 16 * kBlock) DT_ROWB(16, SHORT_ACCESS); \
    else if (row_vecs <= 32 * kBlock) DT_ROWB(32, ACCESS); \
    else DT_ROWB(64, ACCESS);                          \
  } while (0)
  const unsigned wave_grid = (unsigned)ceil_div(rows, kRowsPerBlock);
#define DT_ROW(NV, ACCESS) launcher(rowwise_wave_kernel<IN, OUT, NV, ACCESS>, wave_grid, kBlock, 0, stream)(x, rows, cols, o, amax_out, scale_out)
#define DT_ROW_ANY_LENGTH(ACCESS)                      \
  do {                                                 \
    if (row_vecs <= 1 * kWave) DT_ROW(1, ACCESS);      \
    else if (row_vecs <= 2 * kWave) DT_ROW(2, ACCESS); \
    else if (row_vecs <= 4 * kWave) DT_ROW(4, ACCESS); \
    else if (row_vecs <= 8 * kWave) DT_ROW(8, ACCESS); \
    else DT_ROW(16, ACCESS);                           \
  } while (0)
  if (vec_ok && row_vecs >= block_from && held) {
    DT_ROWB_ANY_LENGTH(kRowsWhole, kRowsWhole);
  } else if (base_ok && !vec_ok && held) {  // rows that are not whole vectors, on an aligned base
    // (few rows: a workgroup each as well, us with a wave and with a workgroup each, fp32: 40 x 1001 2.56 and 2.46,
    // 100 x 1001 2.60 and 2.55, 500 x 1001 2.81 and 2.99, 2000 x 1001 3.93 and 4.39)
    if (row_vecs >= block_from || row_vecs > 16 * kWave || 2 * rows <= device_facts().cu_count) {
      if (edges_cached) DT_ROWB_ANY_LENGTH(kRowsEdges, kRowsEdgesCached);
      else DT_ROWB_ANY_LENGTH(kRowsEdges, kRowsEdges);
    } else if (edges_cached) {
      DT_ROW_ANY_LENGTH(kRowsEdgesCached);
    } else {
      DT_ROW_ANY_LENGTH(kRowsEdges);
    }
  } else if (!vec_ok && held) {  // x or the output not aligned: a workgroup per row with element-aligned vector accesses
    DT_ROWB_ANY_LENGTH(kRowsAny, kRowsAny);
  } else if (vec_ok && row_vecs <= 16 * kWave) {
    DT_ROW_ANY_LENGTH(kRowsWhole);
#undef DT_ROWB
#undef DT_ROWB_ANY_LENGTH
#undef DT_ROW
#undef DT_ROW_ANY_LENGTH
  } else if (vec_ok) {
    launcher(rowwise_block_kernel<IN, OUT, true>, (unsigned)rows, kBlock, 0, stream)(x, cols, o, amax_out, scale_out);
  } else {
    launcher(rowwise_block_kernel<IN, OUT, false>, (unsigned)rows, kBlock, 0, stream)(x, cols, o, amax_out, scale_out);
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
