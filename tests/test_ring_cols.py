"""Tiles of the kernel for few tiles that cover fewer columns than they have, compiled for the host: where their scales are looked for, and which
columns a plan gives them."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS = 256

SOURCE = r"""
#include "mx_gemm_plan.hpp"
#include "mx_ring.hpp"
// The scale words of the tiles of `cols` columns of a matrix of N: every word from where its column's lies (the last one's for those past the
// tile), inside of the descriptor, which does not reach past the matrix.  Returns 0, or what went wrong.
extern "C" int words(int N, int cols, int chunks) {
  for (int n0 = 0; n0 < N; n0 += cols) {
    const int here = N - n0 < cols ? N - n0 : cols;
    for (int step : {0, chunks - 1}) {
      const uint64_t base = (uint64_t)(n0 >> 7) * chunks * 512, all = (uint64_t)((N + 127) / 128) * chunks * 512;
      const uint64_t bytes = (uint64_t)dt::ring_scale_bytes(false, chunks, chunks) + dt::ring_scale_span(n0, here, chunks);
      if (base + bytes > all) return 1;
      for (int w = 0; w < 128; ++w) {
        const uint32_t at = dt::ring_scale_offset(false, w / 64, w % 64, step) + dt::ring_scale_shift(n0, here, chunks, w);
        const int t = (w % 4) * 32 + w / 4, n = n0 + (t < here ? t : here - 1);
        const uint64_t want = ((uint64_t)(n / 128) * chunks + step) * 512 + (n % 32) * 16 + (n % 128) / 32 * 4;
        if (base + at != want) return 2;
        if ((uint64_t)at + 4 > bytes) return 3;
      }
    }
  }
  return 0;
}
extern "C" long plan(int fp4, long M, long N, long K, int ragged, long ws, int cus) {
  const dt::GemmPlan p = dt::plan_gemm(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, 0, false, {3, 1, 0, 0, 0});
  return ((p.small.tile_m * 1000L + p.small.tile_n) * 100 + p.small.splits) * 1000 + p.small.cols;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("ring_cols")
    (where / "cols.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "cols.cpp"), "-o",
                    str(where / "cols.so")], check=True)
    so = C.CDLL(str(where / "cols.so"))
    so.plan.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long, C.c_int]
    so.plan.restype = C.c_long
    return so


def test_scale_words(lib):
    for cols in range(32, 129, 8):
        for N in (4, 8, 60, 128, 132, 1000, 1028, 4096):
            for chunks in (1, 3, 1 << 21):
                assert lib.words(N, cols, chunks) == 0, (N, cols, chunks)


def test_columns(lib):
    def plan(M, N, K, fp4=False):
        rest, cols = divmod(lib.plan(int(fp4), M, N, K, (K // 2 if fp4 else K) % 128 != 0, 1024 + CUS * 65536, CUS), 1000)
        return rest // 100000, rest // 100 % 1000, rest % 100, cols

    assert plan(200, 5120, 5120) == (64, 128, 1, 80) and plan(88, 21328, 8064) == (128, 128, 1, 96)
    assert plan(200, 5120, 5120, True)[3] == 128 and plan(200, 14336, 4096)[3] == 128 and plan(67, 1288, 1280)[3] == 64
    for M in (1, 33, 64, 65, 128, 129, 200, 333, 1000, 4096):
        for N in (4, 8, 1000, 5120, 9304, 21328, 40000):
            for K in (32, 2016, 5120, 16384, 1 << 29):
                tm, tn, splits, cols = plan(M, N, K)
                tiles = -(-M // tm) * -(-N // tn)
                assert cols % 8 == 0 and tn // 2 <= cols <= tn
                if cols != tn:  # a round at most, of more tiles, K in one piece
                    assert splits == 1 and tiles < -(-M // tm) * -(-N // cols) <= CUS and K <= 1 << 28 and N * K >= 8 << 20
