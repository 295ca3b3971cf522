// The block-scaled GEMM for problems of few tiles: out[M,N] = (A 2^sfa)(B 2^sfb)^T with e4m3 or e2m1 operands, tiles of 64 or
// 128 rows and columns, four waves of a quarter of the tile each, K shared between workgroups where tiles are fewer than CUs.
//
// What bounds it is how much a CU may have under way: some 512 requests, whatever their size (measured with LDS-DMA loads of
// 8 rows x 128 bytes: 62 GB/s and CU from memory, 125 from the memory-side cache, however many loads each wave keeps in flight;
// with 16 rows x 64 bytes half of either).  So
//  - every load asks for whole lines: eight lanes per row of a panel, 128 bytes, A and B both through LDS.  (B straight into registers,
//    eight steps ahead, was built: a lane of the MFMA holds 16 bytes of a row, and 128 x 128 tiles took 28 us at
//    200 x 14336 x 4096 where this takes 25.)
//  - a panel's rows are read by the lines they lie in.  Where K is no multiple of 128 bytes a row begins inside a line, and 128 bytes of
//    it from there on would be two requests; here stage w of the ring holds line w of every row (RAGGED), a step's
//    fragments come out of stages w and w + 1, and each lane's addresses say which: a row's phase in its lines is the same for every step.
//    (2048 x 1824 x 1888 e4m3 17.4 -> 14.2 us; 2048 x 1824 x 2048, whole lines, 14.0.)
//  - rows past the matrix are past the end of a buffer descriptor and cost no request (what each load asks for: mx_ring.hpp);
//  - a tile is as small, and K shared as widely, as pays (plan_ring): 64 x 64 tiles ask for half of what 128 x 128 tiles do per step, on
//    four times as many CUs.
// us, 128 x 128 tiles with K shared (what there was) -> here, e4m3 / e2m1, B from memory: 241 x 1336 x 6016 18.7 -> 10.3 / 20.5 ->
// 9.8, 90 x 9304 x 3616 28.3 -> 16.7 / 19.4 -> 11.4, 487 x 3728 x 3872 28.8 -> 17.4 / 18.9 -> 11.8, 256 x 1728 x 1056 9.9 -> 5.7 / 8.5 ->
// 5.3, 512 x 4096 x 4096 22.6 -> 17.7 / 13.6 -> 10.5, 128 x 128 x 16384 23.7 -> 10.1 / 19.4 -> 9.3, 200 x 14336 x 4096 26.1 -> 24.8 /
// 16.4 -> 15.5 (there every CU has a tile already, 264 lines a step: 0.58 us).
//
// A stage of the ring is A's rows, B's rows (128 bytes each) and the scale chunks of one K-step.  Per step one barrier, behind a
// quarter of its MFMAs: every fragment of the step is in registers there, the windows of the next one have landed, and the step's own
// slot is refilled.  Inside a group of 8 rows logical chunk c (16 bytes) of row r sits at position (c + r) % 8, whatever the row's
// phase: a fragment read of 16 rows is free of bank conflicts.  MFMA operands are laid out as in mx_gemm_kernels.hpp.
//
// SPLIT: each share parks its fp32 accumulators in `partial`, lane for lane, and takes a ticket of its tile; whoever draws the last one
// adds the parked accumulators in split order (so the sum does not depend on who came last), writes the bf16 tile and puts the
// ticket counter back to zero.  Nobody waits for anybody.  The parked values travel as device-scope relaxed atomics (stores that
// write through the XCD's L2, loads that miss it): ordinary stores would need a release and an acquire fence around the ticket, i.e. a
// write-back and an invalidation of the whole L2 that every other workgroup of the XCD reads its panels through.
#pragma once

#include <atomic>
#include <type_traits>
#include <utility>

#include "dt_device.hpp"
#include "dt_host.hpp"
#include "mx_gemm_plan.hpp"
#include "mx_ring.hpp"

namespace dt {
namespace ring {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lptr_t;

constexpr int kRingWaves = 4;  // 2 x 2 over the tile

constexpr int stage_bytes(int tm, int tn, bool fp4) { return (tm + tn) * 32 * 128 + 1024 * (fp4 ? 2 : 1); }
// Stages in LDS: as many as fit, an even number.
constexpr int stages(int tm, int tn) { return tm + tn == 4 ? 8 : tm + tn == 6 ? 6 : 4; }

template <typename F, int... I>
__device__ __forceinline__ void each(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <typename F, int... I>
__device__ __forceinline__ bool each_while(F& f, std::integer_sequence<int, I...>) {
  return (f(std::integral_constant<int, I>{}) && ...);
}

// until at most N of this wave's loads are outstanding, and every LDS read has arrived
template <int N>
__device__ __forceinline__ void wait_loads_and_lds() {
  static_assert(N >= 0 && N < 64, "the counter has 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

// TM, TN: 16 x 16 tiles of a wave.  RAGGED: rows that are no whole lines or do not begin on one.  (What the first loads need is the first 14 words
// of the arguments, which are in registers when the kernel begins; lda and ldb are below 2^32 / 255, as the host has checked.  us, with tile counts and
// pitches behind them and both divisions below on every launch -> here, B from memory / from the memory-side cache: e4m3 44 x 4568 x 4672 10.5 -> 10.1 / 8.75 ->
// 8.54, 83 x 6936 x 4384 e2m1 9.96 -> 9.44 / 8.63 -> 8.34; 90 products drawn at random 0.98 / 0.99 of their time, e2m1 0.975 / 0.985.)
// FIT (K not shared): a tile covers fewer columns than it has, in eights, and begins anywhere in a chunk of B's scales; `splits` is 256 times the tiles
// along a row plus the columns of one.
template <int TM, int TN, bool FP4, bool SPLIT, bool RAGGED, bool FIT>
__global__ __launch_bounds__(kRingWaves* kWave) void mx_ring_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, const uint8_t* __restrict__ sfa,
    const uint8_t* __restrict__ sfb, int M, int N, int K, uint32_t lda, uint32_t ldb, int splits, uint16_t* __restrict__ out,
    int64_t ldo, int wide_stores, v4f* __restrict__ partial, uint32_t* __restrict__ tickets) {
#ifdef __HIP_DEVICE_COMPILE__  // the host's pass over this file does not know the registers that the assembly names
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr int KC = FP4 ? 2 : 1;  // 128-element MFMAs (and blocked scale chunks) per K-step
  static_assert((TM == 4 || TM == 2) && (TN == 4 || TN == 2), "tiles of 64 or 128 rows and columns");
  constexpr int kStages = stages(TM, TN), kStageBytes = stage_bytes(TM, TN, FP4);
  constexpr int kOffB = BM * 128, kOffSA = kOffB + BN * 128, kScales = 512 * KC, kOffSB = kOffSA + kScales;
  static_assert(kOffSB + kScales == kStageBytes && kStages % 2 == 0, "a stage: A's rows, B's rows, scale chunks of each");
  constexpr int kLoads = TM + TN + 1;   // per wave and step
  constexpr int kSlots = TM * TN;       // time slots of a step: one e4m3 MFMA or two e2m1 MFMAs each
  constexpr int kBar = kSlots / 4;      // the step's barrier stands behind this slot
  constexpr int kAhead = RAGGED ? 2 : 1;  // a step's fragments lie in its own window and, with RAGGED, in the next one
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave >> 1, wn = wave & 1;

  int bid = blockIdx.x;
  const int tiles_m = (int)((uint32_t)(M + BM - 1) / BM), n_cols = FIT ? splits & 255 : BN;
  const int tiles_n = FIT ? splits >> 8 : (int)((uint32_t)(N + BN - 1) / BN), nb = tiles_m * tiles_n;
  int split = 0;
  if constexpr (SPLIT) {
    split = (int)((uint32_t)bid / (uint32_t)nb);
    bid -= split * nb;
  }
  {  // workgroup b runs on XCD b % 8: each XCD takes a run of neighbouring tiles
    const int q = nb >> 3, r = nb & 7, x = bid & 7;
    bid = x * q + (x < r ? x : r) + (bid >> 3);
  }
  constexpr int kGroup = 8;  // tile rows per group
  int tile_m = 0, tile_n = bid;
  if (tiles_m > 1) {  // (a division in front of the first load is 0.1 us)
    int first_m = 0;
    if (tiles_m > kGroup) {
      const int group = (int)((uint32_t)bid / (uint32_t)(kGroup * tiles_n));
      first_m = group * kGroup;
      bid -= group * kGroup * tiles_n;
    }
    const int gm = (tiles_m - first_m) < kGroup ? (tiles_m - first_m) : kGroup;
    tile_n = (int)((uint32_t)bid / (uint32_t)gm);
    tile_m = first_m + bid - tile_n * gm;
  }
  const int m0 = tile_m * BM, n0 = tile_n * n_cols;
  const int cols = N - n0 < n_cols ? N - n0 : n_cols;

  const int k_bytes = FP4 ? K / 2 : K;
  const int k_steps_all = (k_bytes + kBK - 1) / kBK;
  const int k_chunks = (K + 127) / 128;
  int k_steps = k_steps_all, ks_begin = 0;
  if constexpr (SPLIT) {
    const int per = (int)((uint32_t)(k_steps + splits - 1) / (uint32_t)splits);
    // (scalars, which the compiler cannot tell of what comes out of a division)
    ks_begin = __builtin_amdgcn_readfirstlane(split * per);
    k_steps = __builtin_amdgcn_readfirstlane(k_steps - ks_begin < per ? k_steps - ks_begin : per);
  }
  const int tail_step = k_steps_all - 1 - ks_begin;  // RAGGED: the step whose scales are masked, from ks_begin on
  const int k_windows = k_steps + (RAGGED ? 1 : 0);
  const int left = k_bytes - ks_begin * kBK;  // bytes of a row from ks_begin on

  // ---- memory -> LDS
  struct Operand {
    RingPanel panel;
    v4i rsrc;
    uint32_t bytes;
  };
  auto operand = [&](const uint8_t* first, int rows, uint32_t ld) __attribute__((always_inline)) {
    const uint64_t p = reinterpret_cast<uint64_t>(first), base = RAGGED ? p & ~(uint64_t)127 : p;
    const RingPanel panel{(uint32_t)(p - base), rows, left, ld};
    return Operand{panel, v4i{(int)(uint32_t)base, (int)((uint32_t)(base >> 32) & 0xFFFFu), 0, 0x00027000}, panel.bytes()};
  };
  Operand op_a = operand(A + (uint64_t)m0 * lda + (int64_t)ks_begin * kBK, M - m0 < BM ? M - m0 : BM, lda);
  Operand op_b = operand(B + (uint64_t)n0 * ldb + (int64_t)ks_begin * kBK, cols, ldb);
  uint32_t off_a[TM], off_b[TN], end_a[TM], end_b[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = (wave * TM + i) * 8 + (lane >> 3);
    off_a[i] = op_a.panel.start(RAGGED, r, lane) - (RAGGED ? 0u : i * 1024u);
    end_a[i] = op_a.panel.end(r);
  }
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int r = (wave * TN + i) * 8 + (lane >> 3);
    off_b[i] = op_b.panel.start(RAGGED, r, lane) - (RAGGED ? 0u : i * 1024u);
    end_b[i] = op_b.panel.end(r);
  }
  // Scales: 512 KC bytes of A's chunk row and of B's per step.  e4m3: waves 0, 1 bring the halves of A's chunk, 2 and 3
  // those of B's (4 bytes per lane).  e2m1: even waves bring A's two chunks, odd ones B's (16 bytes per lane,
  // twice the same bytes).
  const bool sc_b = FP4 ? (wave & 1) != 0 : wave >= 2;
  const uint64_t sc_base = reinterpret_cast<uint64_t>(sc_b ? sfb + (int64_t)(n0 >> 7) * k_chunks * 512 : sfa + (int64_t)(m0 >> 7) * k_chunks * 512);
  uint32_t bytes_s = ring_scale_bytes(FP4, k_chunks, ks_begin + k_steps);
  if constexpr (FIT) bytes_s += ring_scale_span(n0, cols, k_chunks) * (uint32_t)(wave >> 1);
  const v4i rsrc_s = v4i{(int)(uint32_t)sc_base, (int)((uint32_t)(sc_base >> 32) & 0xFFFFu), (int)bytes_s, 0x00027000};
  uint32_t off_s = ring_scale_offset(FP4, wave, lane, ks_begin - 1);  // a step is added for each window
  if constexpr (FIT) off_s += ring_scale_shift(n0, cols, k_chunks, (wave & 1) * 64 + lane) * (uint32_t)(wave >> 1);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lptr_t)lds;
  const uint32_t lds_a = lds_base + wave * TM * 1024, lds_b = lds_base + kOffB + wave * TN * 1024;
  const uint32_t lds_s = lds_base + (sc_b ? kOffSB : kOffSA) + (FP4 ? 0 : (wave & 1) * 256);

  // A window past the last one is asked for with empty descriptors (its scales are past the end, or, FIT, others of the matrix that nothing uses): nothing
  // else is read, and the counts stay what they are.
  // Every workgroup walks K front to back, so that an entry is summed in the same order wherever in the matrix it stands.  (With half of
  // the workgroups on runs of K in another order, so that one finds in the XCD's L2 what another one fetched, whole-line products of more than two
  // rows of tiles take 6 to 13 % less from memory and the same from the memory-side cache, us, e4m3 512 x 4096 x 4096 17.7 and 16.2, 400 x 5120 x
  // 5120 28.6 and 25.0, e2m1 300 x 4096 x 8192 17.9 and 16.5; but equal rows of A in different tiles then differ in the last bit.)
  uint32_t at = 0;
  auto aim = [&](int w) __attribute__((always_inline)) {
    const bool in = w < k_windows;
    const RingAsk ask_a = ring_ask(in, op_a.bytes, (uint32_t)w * kBK), ask_b = ring_ask(in, op_b.bytes, (uint32_t)w * kBK);
    op_a.rsrc.z = (int)ask_a.bytes;
    op_b.rsrc.z = (int)ask_b.bytes;
    at = ask_a.at;
    off_s += 512u * KC;
  };
  // load number n of a step into ring slot U: A's groups of 8 rows, B's, the scales.  FIRST: window 0, whose lanes in front of the row
  // read its first chunk.  Of whole lines the groups of a panel go out as a run: the instruction's immediate offset counts in memory
  // and in LDS, lane offsets are lowered by as much (a row is 128 bytes or more, so none goes below zero), and M0, which nothing else
  // here uses, is set once (us, set for each -> once: e2m1 128 x 128 tiles 128 x 8192 x 8192 19.95 -> 19.6, 64 x 64 tiles 12.65 -> 12.5; e4m3 the
  // same within 1 %).
  auto load = [&](auto u_tag, auto n_tag, auto first_tag) __attribute__((always_inline)) {
    constexpr int n = decltype(n_tag)::value, U = decltype(u_tag)::value;
    constexpr bool FIRST = decltype(first_tag)::value;
    if constexpr (n < TM + TN) {
      constexpr bool kA = n < TM;
      constexpr int i = kA ? n : n - TM, kTo = U * kStageBytes + i * 1024;
      const uint32_t to = kA ? lds_a : lds_b;
      uint32_t off = kA ? off_a[kA ? i : 0] : off_b[kA ? 0 : i];
      const v4i r = kA ? op_a.rsrc : op_b.rsrc;
      const uint32_t s = at;
      if constexpr (RAGGED) {
        const uint32_t end = kA ? end_a[kA ? i : 0] : end_b[kA ? 0 : i];
        off += s;
        off = off < end ? off : end;
        if constexpr (FIRST) {
          const uint32_t begin = end + 16 - left;
          off = off > begin ? off : begin;
        }
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     : : "s"(to), "v"(off), "s"(r), "n"(kTo) : "memory", "scc");
      } else if constexpr (i == 0) {
        asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     : : "s"(to), "v"(off), "s"(r), "s"(s), "n"(kTo) : "memory", "scc");
      } else {
        asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%3 lds" : : "v"(off), "s"(r), "s"(s), "n"(i * 1024) : "memory");
      }
    } else {
      constexpr int kTo = U * kStageBytes;
      const uint32_t to = lds_s, off = off_s;
      const v4i r = rsrc_s;
      if constexpr (FP4)
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     : : "s"(to), "v"(off), "s"(r), "n"(kTo) : "memory", "scc");
      else
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                     : : "s"(to), "v"(off), "s"(r), "n"(kTo) : "memory", "scc");
    }
  };

  // ---- fragments and scales of the step in ring slot U
  v8i fa[TM], fb[2][TN];
  int sa[2][KC][TM], sb[2][KC][TN];
  const int kq = lane >> 4, l16 = lane & 15;
  // An LDS instruction's immediate offset spans a few stages: one set of lane addresses for each such window, kept from the
  // compiler's arithmetic (it would work out one per stage and use).  With RAGGED the last slot has one of its own,
  // because the window behind it is slot 0.
  constexpr int kWindow = 65536 / kStageBytes, kSets = (kStages - (RAGGED ? 1 : 0) + kWindow - 1) / kWindow + (RAGGED ? 1 : 0);
  constexpr int kSetOfLast = kSets - 1;
  struct LaneAddresses {
    uint32_t a_lo, a_hi, b_lo, b_hi, s_a, s_b;
  } set[kSets];
  {
    // row l16 of a 16-row tile: group l16 / 8, row l16 % 8; its logical chunk c lies at position (c + l16) % 8, in the step's own window
    // or, c + phase past a line's end, in the next one
    const uint32_t row = (l16 >> 3) * 1024 + (l16 & 7) * 128, lo = row + (((kq + l16) & 7) << 4), hi = lo ^ 64u;
    const uint32_t ph_a = RAGGED ? ((op_a.panel.mis + (uint32_t)(l16 & 7) * lda) & 127u) >> 4 : 0u;
    const uint32_t ph_b = RAGGED ? ((op_b.panel.mis + (uint32_t)(l16 & 7) * ldb) & 127u) >> 4 : 0u;
    const uint32_t a0 = wm * TM * 2048, b0 = kOffB + wn * TN * 2048;
    // even: the first tile's number in its chunk (FIT: B's words come in the order of the tile's columns)
    const int ta = ((m0 & 127) >> 4) + wm * TM, tb = (FIT ? 0 : (n0 & 127) >> 4) + wn * TN;
#pragma unroll
    for (int q = 0; q < kSets; ++q) {
      const bool last = RAGGED && q == kSetOfLast;
      const uint32_t from = (last ? kStages - 1 : q * kWindow) * kStageBytes;
      const uint32_t next = last ? (uint32_t)(-(kStages - 1) * kStageBytes) : (uint32_t)kStageBytes;
      set[q].a_lo = from + a0 + lo + (ph_a + kq >= 8 ? next : 0u);
      set[q].a_hi = from + a0 + hi + (ph_a + kq + 4 >= 8 ? next : 0u);
      set[q].b_lo = from + b0 + lo + (ph_b + kq >= 8 ? next : 0u);
      set[q].b_hi = from + b0 + hi + (ph_b + kq + 4 >= 8 ? next : 0u);
      // the word of row r of a chunk sits at (r % 32) * 16 + (r / 32) * 4, byte = K-block
      set[q].s_a = from + kOffSA + l16 * 16 + kq + (ta >> 1) * 4;
      set[q].s_b = from + kOffSB + l16 * 16 + kq + (tb >> 1) * 4;
      asm volatile("" : "+v"(set[q].a_lo), "+v"(set[q].a_hi), "+v"(set[q].b_lo), "+v"(set[q].b_hi), "+v"(set[q].s_a), "+v"(set[q].s_b));
    }
  }
  auto set_of = [](int slot) { return RAGGED && slot == kStages - 1 ? kSetOfLast : slot / kWindow; };
  auto imm_of = [](int slot) { return RAGGED && slot == kStages - 1 ? 0 : slot % kWindow * kStageBytes; };
  auto read_a = [&](int slot, int i) __attribute__((always_inline)) {
    const LaneAddresses& w = set[set_of(slot)];
    const int o = imm_of(slot) + i * 2048;
    const v4i lo = *reinterpret_cast<const v4i*>(lds + w.a_lo + o), hi = *reinterpret_cast<const v4i*>(lds + w.a_hi + o);
    fa[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto read_b = [&](int slot, int p, int j) __attribute__((always_inline)) {
    const LaneAddresses& w = set[set_of(slot)];
    const int o = imm_of(slot) + j * 2048;
    const v4i lo = *reinterpret_cast<const v4i*>(lds + w.b_lo + o), hi = *reinterpret_cast<const v4i*>(lds + w.b_hi + o);
    fb[p][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto read_scales = [&](int slot, int p) __attribute__((always_inline)) {
    const LaneAddresses& w = set[set_of(slot)];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int o = imm_of(slot) + c * 512;
#pragma unroll
      for (int j = 0; j < TN; ++j) sb[p][c][j] = lds[w.s_b + o + (j & 1) * 256 + (j >> 1) * 4];
#pragma unroll
      for (int i = 0; i < TM; ++i) sa[p][c][i] = lds[w.s_a + o + (i & 1) * 256 + (i >> 1) * 4];
    }
  };
  // RAGGED: the scale bytes of K-blocks past the end of K become 0 on both sides, in the step that holds the last ones
  int lane_mask[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c) lane_mask[c] = kq * 32 + c * 128 < K - (k_steps_all - 1) * 128 * KC ? 0xFF : 0;
  auto settle_scales = [&](int p, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int mask = ks == tail_step ? lane_mask[c] : 0xFF;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (RAGGED) sb[p][c][j] &= mask;
        asm volatile("" : "+v"(sb[p][c][j]));
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if constexpr (RAGGED) sa[p][c][i] &= mask;
        asm volatile("" : "+v"(sa[p][c][i]));
      }
    }
  };

  auto first = [&](auto u_tag) __attribute__((always_inline)) {
    constexpr int U = decltype(u_tag)::value;
    aim(U);
    auto one = [&](auto n_tag) __attribute__((always_inline)) { load(u_tag, n_tag, std::integral_constant<bool, U == 0>{}); };
    each(one, std::make_integer_sequence<int, kLoads>{});
  };
  each(first, std::make_integer_sequence<int, kStages>{});
  // acc becomes zero here, under the first loads.  Each tile's zeros are made values of their own: of one zero for all of them the compiler makes
  // copies in front of the loop, the last of them in the wait states that the first MFMA, whose statement it does not look into, needs behind it.
  v4f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+v"(acc[i][j]));
    }
  wait_loads_and_lds<(kStages - kAhead) * kLoads>();
  __syncthreads();
  read_scales(0, 0);
#pragma unroll
  for (int j = 0; j < TN; ++j) read_b(0, 0, j);
#pragma unroll
  for (int i = 0; i < TM; ++i) read_a(0, i);
  settle_scales(0, 0);

  int ks = 0;
  auto step = [&](auto u_tag) __attribute__((always_inline)) -> bool {
    constexpr int U = decltype(u_tag)::value, P = U & 1, kNext = (U + 1) % kStages;
    __builtin_amdgcn_sched_barrier(0);
    auto slot = [&](auto z_tag) __attribute__((always_inline)) {
      constexpr int z = decltype(z_tag)::value, i = z / TN, j = z % TN;
      if constexpr (!FP4) {
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]"
                     : "+v"(acc[i][j]) : "v"(fb[P][j]), "v"(fa[i]), "v"(sb[P][0][j]), "v"(sa[P][0][i]));
      } else {
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] cbsz:4 blgp:4"
                     : "+v"(acc[i][j]) : "v"(fb[P][j].lo), "v"(fa[i].lo), "v"(sb[P][0][j]), "v"(sa[P][0][i]));
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] cbsz:4 blgp:4"
                     : "+v"(acc[i][j]) : "v"(fb[P][j].hi), "v"(fa[i].hi), "v"(sb[P][KC - 1][j]), "v"(sa[P][KC - 1][i]));
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (z == kBar) {
        // every fragment of this step has been read, so its window's slot is free behind the barrier; the windows of the next
        // step have landed
        wait_loads_and_lds<(kStages - 1 - kAhead) * kLoads>();
        __syncthreads();
        read_scales(kNext, 1 - P);
        aim(ks + kStages);
      }
      if constexpr (z > kBar) {
        constexpr int y = z - kBar - 1, kRest = kSlots - kBar - 1;  // y: 0 .. kRest - 1
        // a[i] is dead behind its last MFMA, slot (i + 1) TN - 1
#pragma unroll
        for (int t = 0; t < TM; ++t)
          if (((t + 1) * TN - 1 > kBar + 1 ? (t + 1) * TN - 1 : kBar + 1) == z) read_a(kNext, t);
#pragma unroll
        for (int t = 0; t < TN; ++t)
          if (t * kRest / TN == y) read_b(kNext, 1 - P, t);
        auto refill = [&](auto n_tag) __attribute__((always_inline)) {
          if constexpr (decltype(n_tag)::value * kRest / kLoads == y) load(u_tag, n_tag, std::false_type{});
        };
        each(refill, std::make_integer_sequence<int, kLoads>{});
        if constexpr (z == kSlots - 2) settle_scales(1 - P, ks + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    each(slot, std::make_integer_sequence<int, kSlots>{});
    return ++ks < k_steps;
  };
  while (each_while(step, std::make_integer_sequence<int, kStages>{})) {
  }
  // what is still on its way lands before the epilogue uses the LDS (the no-ops: an MFMA's result may be read)
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();

  if constexpr (SPLIT) {
    __shared__ uint32_t drawn;
    const int tile_id = tile_m * tiles_n + tile_n;
    const size_t per_split = (size_t)nb * (kRingWaves * TM * TN * kWave);  // accumulators (4 floats each) per split
    uint64_t* const mine = reinterpret_cast<uint64_t*>(partial + ((size_t)tile_id * kRingWaves + wave) * (TM * TN * kWave)) + lane;
    // 16 x 16 tiles wholly outside the matrix are neither parked nor added (uniform per wave); a tile is two planes of 64 x 8 bytes,
    // so that each store instruction writes 512 contiguous bytes
    auto inside = [&](int i, int j) { return m0 + (wm * TM + i) * 16 < M && n0 + (wn * TN + j) * 16 < N; };
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    auto park = [](uint64_t* q, v4f v) {
      const u64x2 w = __builtin_bit_cast(u64x2, v);
      __hip_atomic_store(q, w.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(q + kWave, w.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto fetch_parked = [](const uint64_t* q) -> v4f {
      u64x2 w;
      w.x = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      w.y = __hip_atomic_load(q + kWave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return __builtin_bit_cast(v4f, w);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (inside(i, j)) park(mine + (split * per_split + (i * TN + j) * kWave) * 2, acc[i][j]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the parked values have arrived before the ticket is drawn
    __syncthreads();
    if (tid == 0) drawn = __hip_atomic_fetch_add(tickets + tile_id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (drawn != (uint32_t)(splits - 1)) return;
    if (tid == 0) tickets[tile_id] = 0u;  // every split has drawn: ready for the next launch
    // four shares of half the tile's rows per round trip to memory, added in split order
    constexpr int kBatch = 4, kPart = TM * TN > 8 ? TM / 2 : TM;
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += kPart) {
#pragma unroll
      for (int i = i0; i < i0 + kPart; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
      for (int sp0 = 0; sp0 < splits; sp0 += kBatch) {
        v4f p[kBatch][kPart][TN];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
          for (int i = 0; i < kPart; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              p[u][i][j] = v4f{0.f, 0.f, 0.f, 0.f};
              if (sp0 + u < splits && inside(i0 + i, j))
                p[u][i][j] = fetch_parked(mine + ((sp0 + u) * per_split + ((i0 + i) * TN + j) * kWave) * 2);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
          for (int i = 0; i < kPart; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i0 + i][j] += p[u][i][j];
      }
    }
    __syncthreads();
  }

  // ---- epilogue: bf16 through LDS, whole row segments of 2 BN bytes out
  constexpr int kPitch = BN * 2 + 16;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<u32x2*>(lds + ((wm * TM + i) * 16 + l16) * kPitch + ((wn * TN + j) * 16 + kq * 4) * 2) =
          u32x2{pack_bf16x2(acc[i][j].x, acc[i][j].y), pack_bf16x2(acc[i][j].z, acc[i][j].w)};
  __syncthreads();
  constexpr int kChunks = BN / 8, kRowsPerPass = kRingWaves * kWave / kChunks;
  const int erow = tid / kChunks, echunk = tid % kChunks;
#pragma unroll
  for (int p = 0; p < BM / kRowsPerPass; ++p) {
    const int row = p * kRowsPerPass + erow, m = m0 + row, n = n0 + echunk * 8;
    if (m >= M || n >= N || (FIT && echunk * 8 >= n_cols)) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(lds + row * kPitch + echunk * 16);
    uint16_t* dst = out + (int64_t)m * ldo + n;
    if (wide_stores && n + 8 <= N) {
      *reinterpret_cast<u32x4*>(dst) = v;
    } else {  // N % 4 == 0 is checked on the host: a chunk is 8 or 4 valid columns
      *reinterpret_cast<u32x2*>(dst) = u32x2{v.x, v.y};
      if (n + 8 <= N) *reinterpret_cast<u32x2*>(dst + 4) = u32x2{v.z, v.w};
    }
  }
#endif
}

template <int TM, int TN, bool FP4, bool SPLIT, bool RAGGED, bool FIT = false>
int launch(const RingArgs& p, int splits) {
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr int kLds = stages(TM, TN) * stage_bytes(TM, TN, FP4);
  static_assert(kLds + 64 <= 160 * 1024 && kLds > 82 * 1024 && kLds >= BM * (BN * 2 + 16), "one workgroup per CU; the output tile fits too");
  const int tiles_m = (int)ceil_div(p.M, (int64_t)BM), tiles_n = (int)ceil_div(p.N, (int64_t)(FIT ? p.cols : BN));
  const int64_t grid = (int64_t)tiles_m * tiles_n * splits;
  if (grid > 0x7FFFFFFFll) return DT_ERR_INVALID_SHAPE;
  auto kernel = mx_ring_kernel<TM, TN, FP4, SPLIT, RAGGED, FIT>;
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
  uint8_t* const ws = static_cast<uint8_t*>(p.workspace);
  launcher(kernel, (unsigned)grid, kRingWaves * kWave, kLds, p.stream)(
      p.a, p.b, p.sfa, p.sfb, (int)p.M, (int)p.N, (int)p.K, (uint32_t)p.lda, (uint32_t)p.ldb, FIT ? tiles_n * 256 + p.cols : splits, static_cast<uint16_t*>(p.out), p.ldo,
      (p.ldo % 8 == 0 && aligned(p.out, 16)) ? 1 : 0, ws ? reinterpret_cast<v4f*>(ws + kSplitTicketBytes) : nullptr,
      reinterpret_cast<uint32_t*>(ws));
  return launch_status();
}

template <int TM, int TN, bool FP4>
int launch_tile(const RingArgs& p, bool ragged, int splits) {
  if (splits > 1) return ragged ? launch<TM, TN, FP4, true, true>(p, splits) : launch<TM, TN, FP4, true, false>(p, splits);
  if constexpr (!FP4)
    if (p.cols != 32 * TN) return ragged ? launch<TM, TN, FP4, false, true, true>(p, 1) : launch<TM, TN, FP4, false, false, true>(p, 1);
  return ragged ? launch<TM, TN, FP4, false, true>(p, 1) : launch<TM, TN, FP4, false, false>(p, 1);
}

}  // namespace ring
}  // namespace dt
