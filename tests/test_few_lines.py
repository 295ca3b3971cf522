"""The kernel for at most 32 rows by whole lines, what its addresses are made of, compiled for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include "mx_few_lines.hpp"
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
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("few_lines")
    (where / "f.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "f.cpp"), "-o",
                    str(where / "f.so")], check=True)
    return C.CDLL(str(where / "f.so"))


def test_no_lane_offset_of_b_goes_below_zero(lib):
    for octets in range(1, 9):
        for N in (4, 8, 20, 40, 100, 128, 136, 264, 1000, 2300):
            for k_bytes, ldb in ((128, 128), (128, 256), (256, 256), (384, 512), (8192, 8192), (128, (2**32 - 1 - 3 * 1024 - 128) // 255 // 128 * 128)):
                assert lib.offsets(N, octets, k_bytes, C.c_uint32(ldb)) == 0, (octets, N, ldb)
