"""The rule that picks the kernel of the MXFP4 cast down the columns, compiled on its own for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
COL_T, WIDE, NARROW = range(3)
CUS = 256


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("cast_plan")
    (where / "plan.cpp").write_text(
        '#include "mx_cast_plan.hpp"\n'
        'extern "C" int plan(int f32, int blocked, long rows, long cols, long cus, long pipe_grid, int forced) {\n'
        "  return dt::plan_fp4_cols(f32 != 0, blocked != 0, rows, cols, cus, pipe_grid, forced);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "plan.cpp"), "-o",
                    str(where / "plan.so")], check=True)
    f = C.CDLL(str(where / "plan.so")).plan
    f.argtypes = [C.c_int] * 2 + [C.c_long] * 4 + [C.c_int]
    return lambda rows, cols, f32=False, blocked=True, forced=-1: f(f32, blocked, rows, cols, CUS, 2 * CUS, forced)


# (rows, cols): the kernel that measured best, or within 4 % of it, for (bf16 blocked, bf16 row-major, fp32)
MEASURED = {(512, 512): (NARROW, NARROW, NARROW), (1024, 1664): (NARROW, NARROW, NARROW), (2048, 2048): (NARROW, NARROW, NARROW),
            (32, 15840): (COL_T, COL_T, NARROW), (1152, 6816): (COL_T, COL_T, COL_T), (2432, 3104): (COL_T, COL_T, COL_T),
            (256, 26112): (COL_T, COL_T, COL_T), (3104, 3264): (NARROW, NARROW, NARROW), (672, 14304): (NARROW, NARROW, NARROW),
            (54944, 736): (NARROW, NARROW, NARROW),
            (2560, 3584): (NARROW, NARROW, NARROW), (16608, 704): (COL_T, COL_T, NARROW),
            (12320, 4064): (WIDE, WIDE, NARROW), (15136, 1312): (WIDE, WIDE, NARROW), (44096, 512): (WIDE, WIDE, NARROW),
            (12288, 6144): (WIDE, WIDE, COL_T), (5056, 21056): (NARROW, WIDE, NARROW), (18976, 5376): (NARROW, WIDE, NARROW),
            (16384, 4096): (WIDE, WIDE, COL_T), (8192, 8192): (WIDE, WIDE, COL_T)}


@pytest.mark.parametrize("size", MEASURED, ids=lambda s: f"{s[0]}x{s[1]}")
def test_picks(plan, size):
    bf16, bf16_plain, f32 = MEASURED[size]
    assert plan(*size) == bf16 and plan(*size, blocked=False) == bf16_plain
    assert plan(*size, f32=True) == f32 and plan(*size, f32=True, blocked=False) == f32


def test_forced(plan):
    assert plan(8192, 8192, forced=1) == NARROW and plan(512, 512, forced=0) == COL_T
    assert plan(12544, 6144, forced=0) == WIDE and plan(12544, 6144, f32=True, forced=0) == COL_T
