"""What the loads of the kernel for few tiles ask memory for, compiled for the host: every byte of its operands and scales that a
step uses, and none outside them, whichever way a buffer descriptor's range check treats the scalar offset."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

SOURCE = r"""
#include <vector>
#include "mx_ring.hpp"
namespace {
// does a load of `size` bytes at lane offset v (immediate included) and scalar offset s reach memory?
bool reaches(int rule, uint64_t v, uint32_t s, uint32_t bytes, int size) {
  if (rule == 0) return v + size <= bytes;                                // the scalar offset does not count
  if (rule == 1) return v + s + size <= bytes;                            // it does
  if (rule == 2) return v < (uint32_t)(bytes - s);                        // taken off the number of bytes, which may wrap round
  return (int64_t)v < (int64_t)bytes - (int64_t)s;                        // or not
}
}  // namespace
// One panel of `rows` rows in tiles of `tile` rows, `windows` of its windows and `stages` more.  Returns 0, or what went wrong.
extern "C" int panel(int rule, int ragged, int tile, int rows, int left, long ld, int mis, int windows, int stages) {
  const dt::RingPanel p{(uint32_t)mis, rows, left, ld};
  const uint32_t bytes = p.bytes();
  for (int w = 0; w < windows + stages; ++w) {
    const dt::RingAsk ask = dt::ring_ask(w < windows, bytes, (uint32_t)w * 128);
    std::vector<char> read(bytes + 16, 0);
    for (int r = 0; r < tile; ++r)
      for (int c = 0; c < 8; ++c) {
        const int lane = (r & 7) * 8 + c;
        uint32_t v = p.start(ragged, r, lane), s = ask.at;
        if (ragged) {  // clamped to the row as the kernel does it, the window in the lane offset
          v += (uint32_t)w * 128, s = 0;
          if (v > p.end(r)) v = p.end(r);
          if (w == 0 && v < p.end(r) + 16 - left) v = p.end(r) + 16 - left;
        }
        if (!reaches(rule, v, s, ask.bytes, 16)) continue;
        const uint64_t at = (uint64_t)v + s;
        if (w >= windows) return 1;                                    // past the last window
        if (r >= rows) return 2;                                       // a row that is not there
        if (at < (uint64_t)mis || at + 16 > bytes) return 3;           // outside of the matrix
        if (at < mis + (uint64_t)(r * ld) || at + 16 > mis + (uint64_t)(r * ld) + left) return 4;  // outside of its row
        for (int b = 0; b < 16; ++b) read[at + b] = 1;
      }
    if (w < windows)  // the lines of every row that window w holds, as far as the row goes
      for (int r = 0; r < rows; ++r) {
        const long from = mis + r * ld, line = (from & ~127l) + w * 128l;
        for (long at = line; at < line + 128; ++at)
          if (at >= from && at < from + left && !read[at]) return 5;
      }
  }
  return 0;
}
// The scales of one chunk row of `chunks` chunks for steps begin .. begin + steps - 1, and the windows of `stages` steps more.
extern "C" int scales(int rule, int fp4, int chunks, int begin, int steps, int stages) {
  const uint32_t per = fp4 ? 1024 : 512, bytes = dt::ring_scale_bytes(fp4 != 0, chunks, begin + steps);
  if (bytes > (uint32_t)chunks * 512) return 3;
  for (int w = 0; w < steps + stages; ++w) {
    std::vector<char> read(bytes, 0);
    for (int wave = 0; wave < 2; ++wave)
      for (int lane = 0; lane < 64; ++lane) {
        const uint32_t v = dt::ring_scale_offset(fp4 != 0, wave, lane, begin + w), size = fp4 ? 16 : 4;
        if (!reaches(rule, v, 0, bytes, size)) continue;
        if (w >= steps) return 1;
        if (v + size > bytes) return 3;
        for (uint32_t b = 0; b < size; ++b) read[v + b] = 1;
      }
    for (uint32_t at = (begin + w) * per; w < steps && at < (begin + w + 1) * per && at < (uint32_t)chunks * 512; ++at)
      if (at >= bytes || !read[at]) return 5;
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("ring_loads")
    (where / "loads.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "loads.cpp"), "-o",
                    str(where / "loads.so")], check=True)
    so = C.CDLL(str(where / "loads.so"))
    so.panel.argtypes = [C.c_int] * 5 + [C.c_long] + [C.c_int] * 3
    return so


@pytest.mark.parametrize("rule", range(4))
def test_panels(lib, rule):
    for tile in (64, 128):
        for rows in (1, 7, 8, 63, 64, 65, 127, 128):
            if rows > tile:
                continue
            for k_bytes in (128, 256, 1024, 1152):  # whole lines, one share of K and one of several
                for ld in (k_bytes, k_bytes + 384):
                    for begin in {0, k_bytes // 128 // 2}:
                        left = k_bytes - begin * 128
                        for windows in {1, left // 128}:
                            assert lib.panel(rule, 0, tile, rows, left, ld, 0, windows, 8) == 0, (tile, rows, k_bytes, ld, begin, windows)
            for k_bytes in (16, 32, 112, 144, 1040):  # rows off the lines
                for ld in (k_bytes, k_bytes + 16, k_bytes + 368):
                    for mis in (0, 16, 112):
                        windows = -(-k_bytes // 128) + 1
                        assert lib.panel(rule, 1, tile, rows, k_bytes, ld, mis, windows, 8) == 0, (tile, rows, k_bytes, ld, mis)
                        if k_bytes > 256:
                            assert lib.panel(rule, 1, tile, rows, k_bytes - 256, ld, mis, 3, 8) == 0, (tile, rows, k_bytes, ld, mis)


@pytest.mark.parametrize("rule", range(4))
@pytest.mark.parametrize("fp4", [0, 1], ids=["e4m3", "e2m1"])
def test_scales(lib, rule, fp4):
    for chunks in (1, 2, 3, 8, 9, 33):
        steps_all = -(-chunks // (2 if fp4 else 1))
        for splits in (1, 2, 3):
            per = -(-steps_all // splits)
            for begin in range(0, steps_all, per):
                steps = min(per, steps_all - begin)
                assert lib.scales(rule, fp4, chunks, begin, steps, 9) == 0, (chunks, begin, steps)
