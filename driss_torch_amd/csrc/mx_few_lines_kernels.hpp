// The block-scaled GEMM for at most 32 rows, by whole lines: out[M,N] = (A 2^sfa)(B 2^sfb)^T with e4m3 or e2m1 operands.
//
// Such a problem is one pass over B, and what bounds it beside the memory's rate is how many requests a CU may have under way and how
// many instructions stand between them.  So
//  - every load asks for whole lines, eight rows of 128 bytes straight into LDS, of A and B both (16 bytes per lane in the MFMA's own layout,
//    B straight into registers as in mx_few_rows.hip, are two requests a line);
//  - the scale words of a group of columns lie in as few lines as can be: B's rows come in octets that are neighbours there (octet_column);
//  - a group is 1 to 8 octets wide, so that the groups are one or a few even rounds of the chip: a CU's time is the lines that it asks for
//    (us, B from memory, the kernel for few rows or the small tiles, whichever was the shorter -> here: e4m3 23 x 9928 x 9728, 256 groups of
//    five octets, 23.0 -> 20.8, four octets 27.5; 7 x 10064 x 5856 16.3 -> 13.4; 16 x 28672 x 4096, two rounds of eight, 29.8 -> 22.9);
//  - the waves of a workgroup share K in runs of their own, each with a ring of stages in LDS that no other wave touches, and meet once
//    per group, to add their sums in wave order;
//  - rows that are no whole lines are read by the lines they lie in: a stage holds a window, line w of every row, a step's fragments come out of
//    its window and the one behind it (RAGGED; see mx_ring_kernels.hpp, which lays its panels out the same way): 16 x 8192 x 8160 e4m3
//    19.3 -> 14.9 us, where the requests of half lines straddle them.
// us, before -> here, B from memory / from the memory-side cache: e4m3 16 x 8192 x 8192 16.5 -> 14.4 / 12.9 -> 12.5, 32 x 8192 x 8192 17.6 -> 15.7 /
// 15.7 -> 12.8, 16 x 14336 x 4096 15.0 -> 12.8 / 11.5 -> 11.0, 6 x 3072 x 2048 4.1 -> 3.6 / 3.4 -> 3.0, e2m1 32 x 8192 x 8192 11.4 -> 10.3 / 8.4 -> 7.9.
// 67 MB in 14.4 and 12.5 us is what reading as much takes in any kernel here (amax of 67 MB: 13).  161 problems of 1 to 32 rows drawn at random, both operand
// types, take 0.91 / 0.91 of their time on geometric average.
//
// The order of a step: the fragments of step s are in registers; those of step s + 1 are requested from LDS behind the MFMAs of s, then the loads
// go out that refill the stage of s (a load into LDS leaves a wave every 40 cycles or so), under which those reads arrive.  (Reads, wait, loads,
// MFMAs in turn: about 1000 cycles a step instead of 600; e4m3 15 x 14656 x 5792, four octets, 20.1 -> 19.6 us, from the memory-side cache 17.1 -> 16.5.)
// Where whole lines allow, every wave's run begins at a place of its own and wraps round: with all of them at the same distance from the
// beginning of rows that are a power of two apart, what they ask for at the same time lies in a fraction of the channels (16 x 8192 x
// 8192 e4m3, eight runs of 1024 bytes, 18.5 -> 15.5 us; four of 2048 14.4, so groups of three octets or more have four waves).  The order of an entry's sum is then its column's, the same for every row.
#pragma once

#include <atomic>
#include <type_traits>
#include <utility>

#include "dt_device.hpp"
#include "dt_host.hpp"
#include "mx_few_lines.hpp"

namespace dt {
namespace few_lines {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lptr_t;

template <typename F, int... I>
__device__ __forceinline__ void each(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <typename F, int... I>
__device__ __forceinline__ bool each_while(F& f, std::integer_sequence<int, I...>) {
  return (f(std::integral_constant<int, I>{}) && ...);
}

// MH, NH: octets of A's rows and of a group's columns.  (lda and ldb are below 2^32 / 255, as the host has checked; the arguments that
// the first loads need come first, for the registers that are filled before the kernel begins.)
template <bool FP4, int MH, int NH, bool RAGGED>
__global__ __launch_bounds__(few_lines_waves(FP4, MH, NH, RAGGED) * kWave) void mx_few_lines_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, const uint8_t* __restrict__ sfa, const uint8_t* __restrict__ sfb, int M,
    int N, int K, uint32_t lda, uint32_t ldb, int groups, uint16_t* __restrict__ out, int64_t ldo) {
#ifdef __HIP_DEVICE_COMPILE__  // the host's pass over this file does not know the registers that the assembly names
  constexpr int WAVES = few_lines_waves(FP4, MH, NH, RAGGED);
  constexpr int MT = (MH + 1) / 2, NT = (NH + 1) / 2, KC = FP4 ? 2 : 1;  // 16 x 16 tiles; MFMAs (and scale chunks) per step of 128 bytes
  constexpr bool kOneScaleLoad = few_lines_scales_in_one(MH, NH);
  constexpr int kStages = few_lines_stages_of(WAVES, FP4, MH, NH), kStage = few_lines_stage(FP4, MH, NH), kWaveLds = kStages * kStage;
  constexpr int kOffA = NT * 2048, kOffS = kOffA + MT * 2048;  // a stage: B's rows, A's rows, B's scale words, A's
  constexpr int kOffSA = kOneScaleLoad ? 128 : KC * 256;
  constexpr int kLoads = few_lines_loads(FP4, MH, NH);
  constexpr int kAhead = RAGGED ? 2 : 1;  // a step's fragments lie in its own window and, with RAGGED, in the next one
  static_assert(kStages > kAhead && MT * NT * 1024 <= kStage && (kStages - kAhead) * kLoads < 64, "a ring; a stage holds the wave's sums");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l16 = lane & 15, kq = lane >> 4, lrow = lane >> 3;
  const int k_bytes = FP4 ? K / 2 : K, k_steps = (k_bytes + 127) >> 7, k_chunks = (K + 127) >> 7;
  // this wave's run of steps: the same number of turns for every wave (one without a step of its own loads and adds nothing)
  const int per = (int)((unsigned)(k_steps + WAVES - 1) / (unsigned)WAVES), ks0 = wave * per;
  const int n_steps = ks0 >= k_steps ? 0 : (k_steps - ks0 < per ? k_steps - ks0 : per);
  const int windows = n_steps > 0 ? n_steps + (RAGGED ? 1 : 0) : 0, per_windows = per + (RAGGED ? 1 : 0);
  const int left = k_bytes - ks0 * 128;  // bytes of a row from the run's first step on
  const uint32_t mine = (uint32_t)wave * kWaveLds, lds_wave = (uint32_t)(uintptr_t)(lptr_t)lds + mine;

  // ---- memory -> LDS, through buffer descriptors that begin with the run's first byte and end with the last row's last: a lane in front of
  // the first row (RAGGED: its line begins there) has wrapped round to past the end, and past the end nothing is read.  Lane L brings
  // chunk (16 bytes) L % 8 turned by the row, and by how far into a line the row begins, of row L / 8 of an octet.
  const uint64_t pa = reinterpret_cast<uint64_t>(A) + (uint32_t)ks0 * 128u, pb = reinterpret_cast<uint64_t>(B) + (uint32_t)ks0 * 128u;
  v4i rsrc_a = v4i{(int)(uint32_t)pa, (int)((uint32_t)(pa >> 32) & 0xFFFFu), 0, 0x00027000}, rsrc_b = rsrc_a;
  const uint32_t bytes_a = (uint32_t)(M - 1) * lda + left;
  uint32_t bytes_b = 0;
  const uint32_t mis_a = RAGGED ? (uint32_t)pa & 127u : 0u, mis_b = RAGGED ? (uint32_t)pb & 127u : 0u;  // (octets of rows are whole lines apart)
  auto in_octet = [&](uint32_t mis, uint32_t ld) {
    const uint32_t phase = RAGGED ? (mis + (uint32_t)lrow * ld) & 127u : 0u;
    return ((((uint32_t)lane & 7u) - lrow + (phase >> 4)) & 7u) * 16u - phase;
  };
  const uint32_t in_a = in_octet(mis_a, lda), in_b = in_octet(mis_b, ldb);
  // (whole lines go out in runs of four loads, see few_lines_lane_offset; A's load i is rows 8 i and up, 128 bytes or more each)
  constexpr uint32_t kBias = RAGGED ? 0u : kFewLinesBias;
  uint32_t off_a[MH], off_b[NH];
#pragma unroll
  for (int i = 0; i < MH; ++i) off_a[i] = (uint32_t)(i * 8 + lrow) * lda + in_a - (RAGGED ? 0u : few_lines_immediate(i));
  // scale words: lanes 0 to 31 those of B, the others A's, or 64 of each
  const int arow = kOneScaleLoad ? lane & 31 : lane, arow_in = arow < M ? arow : M - 1;
  const uint64_t sa_lane = reinterpret_cast<uint64_t>(sfa) + (uint32_t)(arow_in & 31) * 16u + (uint32_t)(arow_in >> 5) * 4u;
  uint64_t s_lane = 0;

  // the window to be asked for next: number iw of group ig; at: which step of the run it begins; to_ask: windows that are left to ask for
  const int total = ((groups - 1 - (int)blockIdx.x) / (int)gridDim.x + 1) * per_windows;
  int ig = (int)blockIdx.x - (int)gridDim.x, iw = per_windows, to_ask = total;
  uint32_t at = 0;
  auto enter = [&](int group) __attribute__((always_inline)) {
    const uint32_t first = (uint32_t)group * NH, n0 = (first >> 4) * 128u;
    const uint64_t p = pb + (uint64_t)n0 * ldb - kBias;
    rsrc_b.x = (int)(uint32_t)p;
    rsrc_b.y = (int)((uint32_t)(p >> 32) & 0xFFFFu);
    const int rows = N - (int)n0;
    bytes_b = (uint32_t)((rows < 256 ? rows : 256) - 1) * ldb + left + kBias;  // a group lies in two chunks of 128 rows at most
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      const uint32_t r = few_lines_row(first, i, lrow, (uint32_t)rows);  // (a column that is not there is never stored)
      off_b[i] = RAGGED ? r * ldb + in_b : few_lines_lane_offset(r, ldb, in_b, i);
    }
    const uint32_t i = (uint32_t)(kOneScaleLoad ? lane & 31 : lane) >> 3, octet = first + (i < NH ? i : NH - 1);
    const uint32_t chunks = (uint32_t)(N + 127) >> 7, chunk = (octet >> 4) < chunks ? octet >> 4 : chunks - 1;
    const uint64_t sb_lane = reinterpret_cast<uint64_t>(sfb) + (uint64_t)chunk * ((uint32_t)k_chunks * 512u) + octet_scale_word(octet, lane & 7);
    s_lane = !kOneScaleLoad || lane < 32 ? sb_lane : sa_lane;
    at = RAGGED ? 0u : (((uint32_t)group * 8u + (uint32_t)wave) * 2654435761u >> 16) * (uint32_t)n_steps >> 16;
  };
  // Everything of the next window into a stage, kLoads instructions; nothing behind the last one.  A window behind the end of this wave's run
  // is asked for with empty descriptors (its scale words are those of a step that is there).
  auto issue = [&](uint32_t stage) __attribute__((always_inline)) {
    if (iw == per_windows) {
      iw = 0;
      ig += gridDim.x;
      enter(ig);
    }
    const bool in = iw < windows;
    rsrc_a.z = in ? (int)bytes_a : 0;
    rsrc_b.z = in ? (int)bytes_b : 0;
    const uint32_t step = in ? at : 0u, k = step * 128u, into = lds_wave + stage;
    auto load = [&](auto i_tag, uint32_t to, uint32_t lane_off, v4i r) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value;
      const uint32_t dst = into + to, k_now = k, off = lane_off + k;
      if constexpr (RAGGED)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(dst), "v"(off), "s"(r) : "memory");
      else if constexpr (i % 4 == 0)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(dst), "v"(lane_off), "s"(r), "s"(k_now) : "memory");
      else
        asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%3 lds" : : "v"(lane_off), "s"(r), "s"(k_now), "n"(few_lines_immediate(i)) : "memory");
    };
    auto load_b = [&](auto i) __attribute__((always_inline)) { load(i, decltype(i)::value * 1024, off_b[decltype(i)::value], rsrc_b); };
    auto load_a = [&](auto i) __attribute__((always_inline)) { load(i, kOffA + decltype(i)::value * 1024, off_a[decltype(i)::value], rsrc_a); };
    each(load_b, std::make_integer_sequence<int, NH>{});
    each(load_a, std::make_integer_sequence<int, MH>{});
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      uint32_t chunk = ((uint32_t)ks0 + step) * KC + c;
      chunk = chunk < (uint32_t)k_chunks ? chunk : (uint32_t)k_chunks - 1u;
      const uint64_t so = (uint64_t)(chunk * 512u);  // 4 K bytes at most
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(into + kOffS + c * 256), "v"(s_lane + so) : "memory");
      if constexpr (!kOneScaleLoad)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(into + kOffS + kOffSA + c * 256), "v"(sa_lane + so) : "memory");
    }
    ++at;
    if constexpr (!RAGGED) at = at == (uint32_t)n_steps ? 0u : at;
    ++iw;
  };

  // ---- fragments: chunk c of row l16 of a tile lies at position (c + l16) % 8, in the step's own window or, c + phase past a line's end,
  // in the next one: *_next is all ones there
  const uint32_t row = mine + (l16 >> 3) * 1024 + (l16 & 7) * 128, lane_lo = row + (((kq + l16) & 7) << 4), lane_hi = row + (((kq + 4 + l16) & 7) << 4);
  const uint32_t ph_a = RAGGED ? ((mis_a + (uint32_t)(l16 & 7) * lda) & 127u) >> 4 : 0u, ph_b = RAGGED ? ((mis_b + (uint32_t)(l16 & 7) * ldb) & 127u) >> 4 : 0u;
  const uint32_t a_lo_next = ph_a + kq >= 8 ? ~0u : 0u, a_hi_next = ph_a + kq + 4 >= 8 ? ~0u : 0u;
  const uint32_t b_lo_next = ph_b + kq >= 8 ? ~0u : 0u, b_hi_next = ph_b + kq + 4 >= 8 ? ~0u : 0u;
  const uint32_t lane_s = mine + kOffS + l16 * 4 + kq;  // the lane's byte of row l16's scale word: K-block kq
  v4i a_lo[MT], a_hi[MT], b_lo[NT], b_hi[NT];
  int sa[KC][MT], sb[KC][NT];
  auto read = [&](uint32_t stage, uint32_t next) __attribute__((always_inline)) {  // next: of the window behind it
    const auto place = [&](uint32_t lane_at, uint32_t mask) { return lds + (lane_at + stage + (RAGGED ? mask & (next - stage) : 0u)); };
    const uint8_t *pa_lo = place(lane_lo, a_lo_next) + kOffA, *pa_hi = place(lane_hi, a_hi_next) + kOffA;
    const uint8_t *pb_lo = place(lane_lo, b_lo_next), *pb_hi = place(lane_hi, b_hi_next), *ps = lds + (lane_s + stage);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      b_lo[j] = *reinterpret_cast<const v4i*>(pb_lo + j * 2048);
      b_hi[j] = *reinterpret_cast<const v4i*>(pb_hi + j * 2048);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      a_lo[t] = *reinterpret_cast<const v4i*>(pa_lo + t * 2048);
      a_hi[t] = *reinterpret_cast<const v4i*>(pa_hi + t * 2048);
    }
#pragma unroll
    for (int c = 0; c < KC; ++c) {
#pragma unroll
      for (int j = 0; j < NT; ++j) sb[c][j] = ps[c * 256 + j * 64];
#pragma unroll
      for (int t = 0; t < MT; ++t) sa[c][t] = ps[kOffSA + c * 256 + t * 64];
    }
  };

  v4f acc[MT][NT];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[t][j] = v4f{0.f, 0.f, 0.f, 0.f};
  };
  // The end of a group: the waves park their sums in the stage that each has just used up (the next group's windows are under way into the
  // others), and wave w adds up the tiles w, w + WAVES, ... in wave order and writes them.  (Barriers without the wait for the loads under way.)
  int group = blockIdx.x;
  auto finish = [&](uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<v4f*>(lds + mine + stage + ((t * NT + j) * kWave + lane) * 16) = acc[t][j];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int tile0 = 0; tile0 < MT * NT; tile0 += WAVES) {
      const int tile = tile0 + wave;
      if (tile < MT * NT) {
        v4f sum = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += *reinterpret_cast<const v4f*>(lds + w * kWaveLds + stage + (tile * kWave + lane) * 16);
        const int m = (tile / NT) * 16 + l16, octet = 2 * (tile % NT) + (kq >> 1);
        const uint32_t n = octet_column((uint32_t)group * NH + octet) + 4 * (kq & 1);
        if (m < M && octet < NH && n < (uint32_t)N)  // N % 4 == 0: four columns or none
          *reinterpret_cast<u32x2*>(out + (int64_t)m * ldo + n) = u32x2{pack_bf16x2(sum.x, sum.y), pack_bf16x2(sum.z, sum.w)};
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    clear();
  };

  // Until the loads of `behind` windows are under way and no more, and every LDS read has arrived
  auto wait = [&](int behind) __attribute__((always_inline)) {
    auto exactly = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = kStages - 1 - kAhead - decltype(n_tag)::value;
      if (behind < n) return true;
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(n * kLoads) : "memory");
      return false;
    };
    if (each_while(exactly, std::make_integer_sequence<int, kStages - kAhead>{})) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  };
  // One loop with one copy of everything in it: a launch of few steps spends as much on fetching its instructions as on its data (us, from the
  // memory-side cache, a copy of a step, the end of a group and the loads for each stage -> here: e4m3 6 x 3072 x 2048 3.5 -> 3.0, 23 x 2344 x
  // 2848 5.7 -> 4.3, e2m1 16 x 4096 x 4096 3.5 -> 3.2; long K the same within 2 %).  Turns
  // in front of the first step only ask for windows.  s: the step of the run whose fragments are in registers; with RAGGED a run has one
  // window more than steps, and its turn is the end of the group.
  clear();
  int s = -1;
  uint32_t stage = 0;
  for (int turn = -kStages;; ++turn) {
    const uint32_t next = stage + kStage == kWaveLds ? 0u : stage + kStage;
    if (turn >= -1) {
      // the next step's windows have landed; this one's fragments are in registers, so its stage is free
      const int rest = total - turn;
      wait(rest - 1 - kAhead);
      if (s >= 0 && s < n_steps) {
        if (RAGGED && ks0 + s == k_steps - 1) {  // K-blocks past the end of K: what the rows' last lines hold there counts as nothing, nor do its scales
#pragma unroll
          for (int c = 0; c < KC; ++c) {
            const int keep = kq * 32 + c * 128 < K - (k_steps - 1) * 128 * KC ? -1 : 0;
#pragma unroll
            for (int j = 0; j < NT; ++j) sb[c][j] &= keep;
#pragma unroll
            for (int t = 0; t < MT; ++t) sa[c][t] &= keep;
          }
          const int last = k_bytes - (k_steps - 1) * 128, lo = kq * 16 < last ? -1 : 0, hi = kq * 16 + 64 < last ? -1 : 0;
#pragma unroll
          for (int j = 0; j < NT; ++j) { b_lo[j] &= lo; b_hi[j] &= hi; }
#pragma unroll
          for (int t = 0; t < MT; ++t) { a_lo[t] &= lo; a_hi[t] &= hi; }
        }
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              const v4i zero = {0, 0, 0, 0};
              const v8i vb = FP4 ? __builtin_shufflevector(c == 0 ? b_lo[j] : b_hi[j], zero, 0, 1, 2, 3, 4, 5, 6, 7)
                                 : __builtin_shufflevector(b_lo[j], b_hi[j], 0, 1, 2, 3, 4, 5, 6, 7);
              const v8i va = FP4 ? __builtin_shufflevector(c == 0 ? a_lo[t] : a_hi[t], zero, 0, 1, 2, 3, 4, 5, 6, 7)
                                 : __builtin_shufflevector(a_lo[t], a_hi[t], 0, 1, 2, 3, 4, 5, 6, 7);
              // B as the row operand: a lane holds row l16 of a tile of A and columns 4 kq to 4 kq + 3 of a tile of B
              acc[t][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(vb, va, acc[t][j], FP4 ? 4 : 0, FP4 ? 4 : 0, 0, sb[c][j], 0, sa[c][t]);
            }
      }
      if (rest > 1 && (!RAGGED || s + 1 != per)) read(next, next + kStage == kWaveLds ? 0u : next + kStage);
      ++s;
      if (s == per_windows) {
        finish(stage);
        if (rest == 1) break;
        s = 0;
        group += gridDim.x;
      }
    }
    if (--to_ask >= 0) issue(stage);
    stage = next;
  }
#endif
}

template <bool FP4, int MH, int NH, bool RAGGED>
int launch(const FewLinesArgs& p) {
  constexpr int kWaves = few_lines_waves(FP4, MH, NH, RAGGED);
  constexpr int kLds = kWaves * few_lines_stages_of(kWaves, FP4, MH, NH) * few_lines_stage(FP4, MH, NH);
  static_assert(kLds <= kFewLinesLds && kLds > kFewLinesLds / 2, "one workgroup per CU");
  auto kernel = mx_few_lines_kernel<FP4, MH, NH, RAGGED>;
  static std::atomic<bool> allowed[16];  // once per instantiation and device
  int dev = 0;
  (void)hipGetDevice(&dev);
  const bool tracked = dev >= 0 && dev < 16;
  if (!tracked || !allowed[dev].load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess) {
      (void)hipGetLastError();  // reported here; the next HIP call must not see it again
      return DT_ERR_LAUNCH;
    }
    if (tracked) allowed[dev].store(true, std::memory_order_relaxed);
  }
  const int64_t groups = few_lines_groups(p.N, NH), cus = device_facts().cu_count;
  launcher(kernel, (unsigned)(groups < cus ? groups : cus), kWaves * kWave, kLds, p.stream)(
      p.a, p.b, p.sfa, p.sfb, (int)p.M, (int)p.N, (int)p.K, (uint32_t)p.lda, (uint32_t)p.ldb, (int)groups, static_cast<uint16_t*>(p.out), p.ldo);
  return launch_status();
}

template <bool FP4, int MH, int... NH>
int launch_octets(const FewLinesArgs& p, bool ragged, int octets, std::integer_sequence<int, NH...>) {
  int status = DT_ERR_LAUNCH;
  (void)((octets == NH + 1 && (status = ragged ? launch<FP4, MH, NH + 1, true>(p) : launch<FP4, MH, NH + 1, false>(p), true)) || ...);
  return status;
}
template <bool FP4>
int launch_rows(const FewLinesArgs& p, bool ragged, int octets) {
  constexpr std::make_integer_sequence<int, 8> kOctets{};
  switch ((p.M + 7) / 8) {
    case 1: return launch_octets<FP4, 1>(p, ragged, octets, kOctets);
    case 2: return launch_octets<FP4, 2>(p, ragged, octets, kOctets);
    case 3: return launch_octets<FP4, 3>(p, ragged, octets, kOctets);
    default: return launch_octets<FP4, 4>(p, ragged, octets, kOctets);
  }
}

}  // namespace few_lines
}  // namespace dt
