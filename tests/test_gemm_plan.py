"""The rule that picks the kernel and the tiles of a block-scaled product, compiled on its own for the host: which launch each size
takes, at the sizes where the rule turns."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SMALL, HALVES, T192, T256, THEN_QUADS, THEN_HALVES, QUADRANT_SCHEDULE, FEW_ROWS, FEW_LINES = range(9)
CUS = 256
ALL = 1024 + CUS * 128 * 128 * 4  # a workspace with room for a tile per CU


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text(
        '#include "mx_gemm_plan.hpp"\n'
        'extern "C" int plan(int fp4, long M, long N, long K, int ragged, long ws, int cus, int few, int variant, int tail, int split_k) {\n'
        "  const dt::GemmPlan p = dt::plan_gemm(fp4 != 0, M, N, K, ragged != 0, (size_t)ws, cus, few, few && dt::few_lines_fits(M, K), {variant, tail, split_k, 0, 0});\n"
        "  return p.tiles * 100 + p.small.splits;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "plan.cpp"), "-o",
                    str(where / "plan.so")], check=True)
    f = C.CDLL(str(where / "plan.so")).plan
    f.argtypes = [C.c_int] + [C.c_long] * 3 + [C.c_int, C.c_long] + [C.c_int] * 5

    def call(fp4, M, N, K, ws=ALL, cus=CUS, variant=0, tail=1, split_k=0, few=0):
        return divmod(f(int(fp4), M, N, K, (K // 2 if fp4 else K) % 128 != 0, ws, cus, few, variant, tail, split_k), 100)

    return call


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("size,tiles", [
    # a quarter to half a round of 256 x 256 tiles: one round of 128 x 128 tiles where that is enough ...
    ((65, 16648), SMALL), ((96, 28672), SMALL), ((128, 32512), SMALL), ((300, 10000), SMALL), ((1152, 3584), SMALL),
    # ... also at exactly half a round of the large tiles, with half of each outside the matrix, and mirrored
    ((65, 32520), SMALL), ((128, 32768), SMALL), ((32768, 128), SMALL), ((32700, 65), SMALL),
    # one column more is two rounds of them, but one of 256 x 192 tiles
    ((128, 32776), T192), ((128, 49152), T192), ((128, 49160), T256),
    # halves where 128 x 128 tiles do not fit
    ((129, 16648), HALVES), ((256, 32768), HALVES), ((2048, 4096), HALVES), ((300, 14336), HALVES), ((2048, 2048), SMALL),
    ((2304, 2304), HALVES),
    # more than half a round
    ((2048, 4352), T192), ((2000, 6144), T192), ((2048, 6400), T256), ((4096, 4096), T256),
    # whole rounds and what is left over
    ((4096, 5120), THEN_QUADS), ((4096, 6144), THEN_HALVES), ((4096, 6400), T256), ((8192, 8192), T256)], ids=str)
def test_tiles_by_size(plan, fp4, size, tiles):
    assert plan(fp4, *size, 1024)[0] == tiles


def test_one_round_of_small_tiles_is_never_given_to_fewer_large_ones(plan):
    """wherever 128 x 128 tiles are one round, a plan of larger ones has to keep more than half of the chip busy"""
    for rows in (64, 65, 128, 129, 256, 300, 640, 1152, 2048, 4096, 20000, 32768):
        for n in range(128, 60000, 248):
            for m, n_ in ((rows, n), (n, rows)):
                up = lambda a, b: -(-a // b)  # noqa: E731
                if up(m, 128) * up(n_, 128) <= CUS:
                    assert plan(False, m, n_, 1024)[0] == SMALL, (m, n_)


def test_knobs(plan):
    assert plan(False, 2048, 6144, 1024, variant=1) == (SMALL, 1) and plan(False, 128, 128, 16384, variant=1)[1] > 1
    assert plan(False, 16, 64, 1024, variant=2)[0] == T256
    assert plan(False, 16, 64, 1024, variant=5)[0] == T192
    assert plan(False, 16, 64, 1024, variant=7)[0] == QUADRANT_SCHEDULE
    assert plan(False, 4096, 5120, 1024, tail=0)[0] == T256 and plan(False, 2048, 4096, 1024, tail=0)[0] == T256
    assert plan(False, 4096, 5120, 1024, tail=3)[0] == THEN_HALVES and plan(False, 4096, 6400, 1024, tail=2)[0] == THEN_QUADS


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
def test_rows_off_the_lines_take_small_tiles_instead_of_halves(plan, fp4):
    """from 385 rows and 16 steps on, the last of them partly filled"""
    step = 256 if fp4 else 128
    for M, N in ((384, 12008), (385, 12008), (400, 8200), (726, 9072), (2048, 4096)):
        for steps in (2, 15, 16, 17, 64):
            K = (steps - 1) * step + 32
            assert plan(fp4, M, N, K)[0] == (SMALL if M > 384 and steps > 15 else HALVES), (M, N, steps)
            assert plan(fp4, M, N, steps * step)[0] == HALVES


def test_few_rows(plan):
    for M in (1, 16, 32, 33, 48):
        assert plan(True, M, 2048, 4096, few=16)[0] == (FEW_LINES if M <= 32 else FEW_ROWS) and plan(True, M, 2048, 4096)[0] == SMALL
        assert plan(False, M, 64, 128, few=16, variant=9)[0] == (FEW_LINES if M <= 32 else FEW_ROWS)
    assert plan(False, 100, 64, 64, variant=9)[0] == SMALL
    for variant, tiles in ((1, SMALL), (2, T256), (3, SMALL), (5, T192), (7, QUADRANT_SCHEDULE)):
        for M in (16, 40):
            assert plan(False, M, 8192, 8192, few=32, variant=variant)[0] == tiles


def test_short_rows_off_the_lines_keep_the_kernel_that_loads_b_into_registers(plan):
    """of at most 32 rows, those of up to 16 columns per CU and of few steps"""
    for fp4, M, steps in ((True, 1, 16), (True, 16, 16), (True, 17, 24), (True, 32, 24), (False, 16, 16), (False, 17, 16), (False, 32, 16)):
        step = 256 if fp4 else 128
        for N in (8, 1024, 4096):
            for n, off in ((steps, 32), (steps + 1, 32), (steps, step)):
                few = plan(fp4, M, N, (n - 1) * step + off, few=16)[0]
                assert few == (FEW_ROWS if n == steps and off == 32 else FEW_LINES), (fp4, M, N, n, off)
        assert plan(fp4, M, 4104, (steps - 1) * step + 32, few=16, variant=9)[0] == FEW_LINES
        assert plan(fp4, M, 4104, steps * step, few=16, variant=10)[0] == FEW_ROWS
    assert plan(False, 16, 1024, 9 * 128 - 96, few=16)[0] == FEW_ROWS and plan(False, 16, 1024, 8 * 128 - 96, few=16)[0] == FEW_LINES
    assert plan(False, 17, 1024, 32, few=16)[0] == FEW_ROWS and plan(True, 1, 1024, 32, few=16)[0] == FEW_ROWS


def test_shares_own_a_step_and_fit_the_workspace(plan):
    for fp4 in (False, True):
        for K in (32, 256, 288, 1024, 5152, 16416, 65536):
            steps = -(-K // (256 if fp4 else 128))
            for M, N in ((1, 8), (128, 128), (300, 264), (1024, 1024), (128, 16384)):
                tiles = -(-M // 128) * -(-N // 128)
                for split_k in (0, 2, 3, 5, 16, 99):
                    for room in (1, tiles, 2 * tiles + 1, 256):
                        n = plan(fp4, M, N, K, ws=1024 + room * 128 * 128 * 4, split_k=split_k, variant=1)[1]
                        assert 1 <= n <= 16 and (n == 1 or n * tiles <= room)
                        assert (n - 1) * -(-steps // n) < steps  # the last share owns a step
