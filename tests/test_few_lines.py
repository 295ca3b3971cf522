"""The kernel for at most 32 rows by whole lines, compiled for the host: what its addresses are made of, its ring, and the form that the estimate picks."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include <vector>
#include "mx_gemm_plan.hpp"
// The loads of B by whole lines, every group of `octets` octets of N columns: the descriptor begins kFewLinesBias bytes in front of the group's
// first chunk and ends with its last row.  Returns 0, or what is wrong with an offset: 1 lane and immediate offset do not add up to the
// bytes of the column without going below zero, 2 they end past the last row, 3 another column's.
extern "C" int offsets(int N, int octets, uint32_t k_bytes, uint32_t ldb) {
  for (uint32_t group = 0; group < dt::few_lines_groups(N, octets); ++group) {
    const uint32_t first = group * octets, n0 = (first >> 4) * 128u, rows = N - n0;
    const uint64_t bytes = (uint64_t)((rows < 256 ? rows : 256) - 1) * ldb + k_bytes + dt::kFewLinesBias;
    for (int i = 0; i < octets; ++i)
      for (uint32_t lane = 0; lane < 64; ++lane) {
        const uint32_t r = dt::few_lines_row(first, i, lane >> 3, rows), n = dt::octet_column(first + i) + (lane >> 3);
        if (n0 + r != (n < (uint32_t)N ? n : (uint32_t)N - 1)) return 3;
        const uint32_t in_row = (lane & 7) * 16;  // (turned by the row: some lane of the row has each of them)
        const uint64_t at = (uint64_t)dt::few_lines_lane_offset(r, ldb, in_row, i) + dt::few_lines_immediate(i);
        if (at != (uint64_t)dt::kFewLinesBias + (uint64_t)r * ldb + in_row) return 1;
        if (at + 16 + k_bytes - 128 > bytes) return 2;
      }
  }
  return 0;
}
// Every column of N in exactly one octet of exactly one group, no group behind the last chunk of 128 columns, the scale word of each where the
// blocked layout has that row's.  Returns 0, or what is wrong.
extern "C" int octets(int N, int octets) {
  std::vector<int> seen(N, 0);
  for (uint32_t group = 0; group < dt::few_lines_groups(N, octets); ++group) {
    if (dt::octet_column(group * octets) / 128 > (uint32_t)(N - 1) / 128) return 3;
    for (uint32_t octet = group * octets; octet < (group + 1) * octets; ++octet)
      for (uint32_t row = 0; row < 8; ++row) {
        const uint32_t n = dt::octet_column(octet) + row;
        if (n / 128 != octet / 16) return 1;
        if ((octet / 16) * 512 + dt::octet_scale_word(octet, row) != (n / 128) * 512 + (n % 32) * 16 + n % 128 / 32 * 4) return 2;
        if (n < (uint32_t)N) ++seen[n];
      }
  }
  for (int n : seen)
    if (n != 1) return 4;
  return 0;
}
extern "C" int ring(int fp4, int mh, int nh, int ragged, int* waves, int* loads, int* bytes) {
  *waves = dt::few_lines_waves(fp4, mh, nh, ragged);
  *loads = dt::few_lines_loads(fp4, mh, nh);
  *bytes = dt::few_lines_stage(fp4, mh, nh);
  return dt::few_lines_stages_of(*waves, fp4, mh, nh);
}
extern "C" long plan(int fp4, long M, long N, long K, int forced, int cus) {
  const dt::FewLinesPlan p = dt::plan_few_lines(fp4 != 0, M, N, K, (fp4 ? K / 2 : K) % 128 != 0, cus, forced);
  return p.ns * 10 + p.octets;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("few_lines")
    (where / "f.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "f.cpp"), "-o",
                    str(where / "f.so")], check=True)
    so = C.CDLL(str(where / "f.so"))
    so.plan.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int] * 2
    so.plan.restype = C.c_long
    return so


def test_no_lane_offset_of_b_goes_below_zero(lib):
    for octets in range(1, 9):
        for N in (4, 8, 20, 40, 100, 128, 136, 264, 1000, 2300):
            for k_bytes, ldb in ((128, 128), (128, 256), (256, 256), (384, 512), (8192, 8192), (128, (2**32 - 1 - 3 * 1024 - 128) // 255 // 128 * 128)):
                assert lib.offsets(N, octets, k_bytes, C.c_uint32(ldb)) == 0, (octets, N, ldb)


def test_octets_hold_every_column_once(lib):
    for octets in range(1, 9):
        for N in (4, 8, 20, 36, 100, 128, 136, 264, 1000, 2300, 8192):
            assert lib.octets(N, octets) == 0, (octets, N)


def test_rings_fit_the_lds_and_the_counter_of_loads(lib):
    for fp4 in (0, 1):
        for mh in range(1, 5):
            for nh in range(1, 9):
                for ragged in (0, 1):
                    waves, loads, stage = C.c_int(), C.c_int(), C.c_int()
                    stages = lib.ring(fp4, mh, nh, ragged, C.byref(waves), C.byref(loads), C.byref(stage))
                    assert waves.value in (2, 4, 8) and stages * waves.value * stage.value <= 160 * 1024
                    assert stages >= (3 if ragged else 2)  # a step's windows, and one under way besides them
                    assert (stages - 1) * loads.value <= 63 and stages * stage.value <= 1 << 16  # 6 and 16 bits
                    tiles = (mh + 1) // 2 * ((nh + 1) // 2)
                    assert stage.value >= tiles * 1024  # the wave's sums are parked in one


def test_octets_by_size(lib):
    def octets(M, N, K, fp4=0, forced=0, cus=256):
        return lib.plan(fp4, M, N, K, forced, cus) % 10

    # a group per CU where that is one round, as many even rounds as the widest groups take beyond it
    assert octets(16, 8192, 8192) == 4 and octets(32, 8192, 8192, 1) == 4 and octets(23, 9928, 9728) == 5 and octets(7, 10064, 5856) == 5
    assert octets(6, 3072, 2048) == 2 and octets(1, 1024, 4096) == 1 and octets(16, 28672, 4096) == 7
    for M in (1, 8, 9, 16, 31, 32):
        for N in (4, 64, 2048, 3000, 28672, 1 << 20):
            for K in (32, 96, 4096, 16416, 1 << 29):
                for fp4 in (0, 1):
                    assert 1 <= octets(M, N, K, fp4) <= 8 and lib.plan(fp4, M, N, K, 0, 256) > 0
                    for forced in (1, 5, 8):
                        assert octets(M, N, K, fp4, forced) == forced
                        assert lib.plan(fp4, M, N, K, 0, 256) // 10 <= lib.plan(fp4, M, N, K, forced, 256) // 10  # the shortest of all
