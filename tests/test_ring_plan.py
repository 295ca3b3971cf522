"""The estimate that picks the small tiles of a block-scaled product, the workgroups that share K and the kernels for few
rows, compiled on its own for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS = 256
ALL = 1024 + CUS * 128 * 128 * 4

# (M, K, N): tile and workgroups that share its K, e4m3 and e2m1; the GPU tests compute the same products
SHARES = {(256, 8192, 8192): ((64, 128, 1), (64, 128, 1)),
          (250, 7200, 8184): ((64, 128, 1), (64, 128, 1)),
          (256, 16384, 8192): ((128, 128, 2), (64, 128, 1)),
          (100, 4128, 14336): ((128, 64, 1), (128, 64, 1)),
          (128, 5120, 5120): ((64, 64, 1), (64, 64, 1)),
          (65, 5152, 5000): ((128, 64, 3), (64, 64, 1)),
          (200, 5120, 5120): ((64, 128, 1), (64, 128, 1)),
          (128, 8192, 8192): ((64, 64, 1), (64, 64, 1)),
          (120, 8064, 8184): ((64, 64, 1), (64, 64, 1)),
          (128, 8096, 8000): ((64, 64, 1), (64, 64, 1)),
          (128, 16416, 4096): ((64, 128, 4), (64, 64, 2)),
          (256, 4096, 4096): ((64, 64, 1), (64, 64, 1)),
          (1000, 2048, 2048): ((64, 128, 1), (64, 128, 1)),
          (71, 12544, 5688): ((128, 128, 5), (128, 64, 2)),
          (195, 6144, 4144): ((128, 128, 3), (64, 128, 1)),
          (72, 8704, 5128): ((128, 64, 3), (64, 64, 1)),
          (67, 13824, 2488): ((128, 64, 6), (64, 64, 3)),
          (578, 13056, 744): ((64, 128, 4), (64, 64, 2)),
          (325, 11520, 1536): ((64, 128, 3), (64, 128, 3)),
          (455, 4352, 192): ((64, 64, 5), (64, 64, 2)),
          (91, 12288, 272): ((64, 64, 12), (64, 64, 8)),
          (200, 5952, 4960): ((128, 128, 3), (64, 128, 1)),
          (73, 13408, 5520): ((128, 128, 5), (128, 64, 2)),
          (72, 12512, 3488): ((128, 64, 4), (64, 64, 2)),
          (99, 9184, 3704): ((128, 64, 4), (64, 64, 2)),
          (162, 11936, 1800): ((64, 128, 5), (64, 64, 2)),
          (229, 10208, 1528): ((64, 128, 5), (64, 64, 2)),
          (251, 14656, 992): ((64, 64, 4), (64, 64, 4)),
          (380, 7616, 208): ((64, 64, 6), (64, 64, 5)),
          (76, 12288, 5392): ((128, 64, 3), (128, 64, 3)),
          (785, 11264, 616): ((64, 128, 3), (64, 128, 3)),
          (585, 12352, 816): ((128, 64, 3), (128, 64, 3)),
          (96, 11296, 4216): ((128, 64, 3), (128, 64, 3)),
          (654, 11232, 784): ((64, 128, 3), (64, 128, 3)),
          (151, 13760, 2784): ((64, 128, 3), (64, 128, 3))}


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("ring_plan")
    (where / "plan.cpp").write_text(
        '#include "mx_gemm_plan.hpp"\n'
        'extern "C" long ring(int fp4, long M, long N, long K, int ragged, long ws, int cus, int split_k, int tm, int tn) {\n'
        "  const dt::RingPlan p = dt::plan_ring(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, split_k, tm, tn);\n"
        "  return (p.tile_m * 1000L + p.tile_n) * 100 + p.splits;\n}\n"
        'extern "C" int few(int fp4, long M, long N, long K, int ragged, long ws, int cus, int columns, int split_k) {\n'
        "  const dt::GemmTiles t = dt::plan_gemm(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, columns, dt::few_lines_fits(M, K), {0, 1, split_k, 0, 0}).tiles;\n"
        "  return t == dt::kFewRows || t == dt::kFewLines;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "plan.cpp"), "-o",
                    str(where / "plan.so")], check=True)
    so = C.CDLL(str(where / "plan.so"))
    so.ring.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long] + [C.c_int] * 4
    so.ring.restype = C.c_long
    so.few.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long] + [C.c_int] * 3
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

    def few(M, N, K, fp4=0, split_k=0):
        return lib.few(fp4, M, N, K, (K // 2 if fp4 else K) % 128 != 0, ALL, CUS, 32 if N >= 8192 else 16, split_k)

    assert few(16, 8192, 8192) and few(1, 1928, 1984) and few(16, 4096, 4096, 1)
    assert few(1, 168, 10048, 1) and few(12, 1488, 12064, 1) and few(2, 464, 5152) and not few(64, 424, 8224)
    for split_k in (1, 2, 7):  # how many workgroups share K says nothing about the kernels for few rows; that none may can only speak for them
        assert few(16, 8192, 8192, split_k=split_k) and few(16, 4096, 4096, 1, split_k) and few(40, 4096, 4096, split_k=split_k)
    assert few(40, 1024, 8192, split_k=1) and not few(40, 1024, 8192, split_k=2) and not few(40, 1024, 8192)
    assert few(16, 1024, 8192) and few(16, 5120, 5120)  # at most 32 rows: by whole lines
    assert not few(64, 8192, 8192) and not few(32, 28672, 10848) and not few(32, 14336, 4096, 1)


@pytest.mark.parametrize("size", SHARES, ids=lambda s: "x".join(map(str, s)))
def test_shares_of_k(lib, size):
    M, K, N = size
    for fp4 in (False, True):
        assert ring(lib, M, N, K, fp4) == SHARES[size][fp4]
        assert ring(lib, M, N, K, fp4, ws=0)[2] == 1 and ring(lib, M, N, K, fp4, split_k=1)[2] == 1


def test_the_sizes_above_share_k_in_every_way():
    """even and uneven shares of whole lines and of rows off them, on every tile that the rule shares"""
    seen = set()
    for (M, K, N), plans in SHARES.items():
        for fp4 in (False, True):
            tm, tn, n = plans[fp4]
            k_bytes = K // 2 if fp4 else K
            if n > 1:
                seen.add((fp4, (tm, tn), k_bytes % 128 != 0, -(-k_bytes // 128) % n == 0))
    for ragged in (False, True):
        for even in (False, True):
            for tile in ((64, 64), (64, 128), (128, 64), (128, 128)):
                assert (False, tile, ragged, even) in seen, (tile, ragged, even)
                assert (True, tile, ragged, even) in seen or tile == (128, 128), (tile, ragged, even)  # e2m1: smaller tiles are shorter
