"""The estimate that picks the small tiles of a block-scaled product, the workgroups that share K and the kernel for few
rows, compiled on its own for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS = 256
ALL = 1024 + CUS * 128 * 128 * 4


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("ring_plan")
    (where / "plan.cpp").write_text(
        '#include "mx_gemm_plan.hpp"\n'
        'extern "C" long ring(int fp4, long M, long N, long K, int ragged, long ws, int cus, int split_k, int tm, int tn) {\n'
        "  const dt::RingPlan p = dt::plan_ring(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, split_k, tm, tn);\n"
        "  return (p.tile_m * 1000L + p.tile_n) * 100 + p.splits;\n}\n"
        'extern "C" int few(int fp4, long M, long N, long K, int ragged, long ws, int cus, int columns) {\n'
        "  const dt::RingPlan p = dt::plan_ring(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, 0, 0, 0);\n"
        "  return dt::few_rows_beats(p, fp4 != 0, M, N, K, ragged != 0, cus, columns);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "plan.cpp"), "-o",
                    str(where / "plan.so")], check=True)
    so = C.CDLL(str(where / "plan.so"))
    so.ring.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long] + [C.c_int] * 4
    so.ring.restype = C.c_long
    so.few.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long] + [C.c_int] * 2
    return so


def ring(lib, M, N, K, fp4=False, ws=ALL, split_k=0, tile=(0, 0)):
    r = lib.ring(int(fp4), M, N, K, (K // 2 if fp4 else K) % 128 != 0, ws, CUS, split_k, *tile)
    return r // 100000, r // 100 % 1000, r % 100


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
def test_every_share_owns_a_step_and_the_workspace_holds_them(lib, fp4):
    for K in (32, 256, 288, 1024, 5152, 16416, 65536, 1 << 24):
        steps = -(-K // (256 if fp4 else 128))
        for M, N in ((1, 8), (64, 128), (129, 128), (300, 264), (1024, 1024), (128, 16384), (40, 200000), (8192, 8192)):
            for tile in ((0, 0), (64, 64), (64, 128), (128, 64), (128, 128)):
                for split_k in (0, 1, 2, 5, 99):
                    for ws in (0, 1024, 1024 + 65536, ALL):
                        tm, tn, n = ring(lib, M, N, K, fp4, ws, split_k, tile)
                        assert (tm, tn) == tile if tile[0] else tm in (64, 128) and tn in (64, 128)
                        tiles = -(-M // tm) * -(-N // tn)
                        assert 1 <= n <= 16 and (n == 1 or (n * tiles * tm * tn * 4 + 1024 <= ws and tiles <= 256))
                        assert (n - 1) * -(-steps // n) < steps and (split_k != 1 or n == 1)


def test_picks(lib):
    # (M, N, K): the form that measured best, or within 2 % of it, B from memory
    assert ring(lib, 200, 14336, 4096) == (128, 128, 1)  # smaller tiles would be two rounds of the chip
    assert ring(lib, 128, 14336, 4096)[2] == 1 and ring(lib, 256, 1728, 1056) == (64, 64, 1)
    assert ring(lib, 128, 128, 16384)[2] >= 8  # four tiles: K shared as widely as it goes
    assert ring(lib, 128, 8192, 8192) == (64, 64, 1) and ring(lib, 384, 1024, 8192) == (64, 64, 2)  # parking 128 x 128 tiles costs more
    assert ring(lib, 512, 512, 16384) == (64, 64, 4) and ring(lib, 2048, 1824, 1888) == (128, 128, 1)
    few = lambda M, N, K, fp4=0: lib.few(fp4, M, N, K, (K // 2 if fp4 else K) % 128 != 0, ALL, CUS, 32 if N >= 8192 else 16)  # noqa: E731
    assert few(16, 8192, 8192) and few(1, 1928, 1984) and few(16, 4096, 4096, 1)
    assert not few(64, 8192, 8192) and not few(32, 28672, 10848) and not few(32, 14336, 4096, 1) and not few(16, 5120, 5120)
