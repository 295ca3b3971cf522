"""The rules that pick the tiles of the MXFP8 cast and the kernel of the MXFP4 cast down the columns and the tile order of the casts along both
axes, compiled on their own for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
COL_T, WIDE, NARROW = range(3)
CUS = 256


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("cast_plan")
    (where / "plan.cpp").write_text(
        '#include "mx_cast_plan.hpp"\n'
        'extern "C" int plan(int f32, int blocked, long rows, long cols, long cus, long pipe_grid, int forced) {\n'
        "  return dt::plan_fp4_cols(f32 != 0, blocked != 0, rows, cols, cus, pipe_grid, forced);\n}\n"
        'extern "C" int narrow_cols(int f32, int blocked, long rows, long cols, long cus) {\n'
        "  return dt::narrow_cols(f32 != 0, blocked != 0, rows, cols, cus);\n}\n"
        'extern "C" int order(int f32, int fp4, int narrow, long rows, long cols, long cus) {\n'
        "  return dt::pair_order(f32 != 0, fp4 != 0, narrow != 0, rows, cols, cus);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'driss_torch_amd' / 'csrc'}", str(where / "plan.cpp"), "-o",
                    str(where / "plan.so")], check=True)
    so = C.CDLL(str(where / "plan.so"))
    so.plan.argtypes = [C.c_int] * 2 + [C.c_long] * 4 + [C.c_int]
    so.narrow_cols.argtypes = [C.c_int] * 2 + [C.c_long] * 3
    so.order.argtypes = [C.c_int] * 3 + [C.c_long] * 3
    return so


@pytest.fixture(scope="module")
def plan(lib):
    return lambda rows, cols, f32=False, blocked=True, forced=-1: lib.plan(f32, blocked, rows, cols, CUS, 2 * CUS, forced)


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


@pytest.mark.parametrize("f32,fp4,narrow,size,order", [
    (0, 0, 0, (16384, 4096), 1), (0, 0, 1, (8192, 8192), 1), (0, 0, 1, (4096, 14336), 1), (0, 0, 1, (2976, 11968), 0), (0, 0, 1, (3040, 11968), 1),
    (1, 0, 0, (3840, 10784), 1), (1, 0, 0, (3584, 8192), 0), (1, 1, 0, (3584, 8192), 0), (1, 0, 0, (4096, 16384), 1), (0, 1, 0, (3584, 8192), 1),
    (0, 1, 0, (16384, 2560), 2), (1, 1, 0, (8192, 2560), 2), (0, 0, 0, (16384, 2560), 1), (0, 1, 0, (14336, 1024), 1), (0, 1, 0, (3040, 6528), 1)])
def test_order_of_the_casts_along_both_axes(lib, f32, fp4, narrow, size, order):
    assert lib.order(f32, fp4, narrow, *size, CUS) == order


@pytest.mark.parametrize("f32,blocked,size,narrow", [
    (0, 1, (512, 512), 1), (0, 0, (2752, 4096), 1), (0, 1, (4096, 3488), 0), (0, 0, (6144, 4096), 0), (0, 1, (3584, 8192), 1), (0, 1, (8192, 8192), 1),
    (0, 1, (6240, 11968), 1), (0, 0, (6240, 11968), 0), (0, 1, (16384, 4096), 1), (0, 0, (16384, 4096), 0), (0, 0, (14336, 4096), 1),
    (1, 1, (512, 512), 1), (1, 0, (2048, 4096), 1), (1, 1, (4096, 4096), 0), (1, 1, (8192, 8192), 0),
    (1, 1, (16384, 64), 1), (1, 1, (20480, 64), 0), (1, 0, (20480, 64), 1), (1, 1, (65536, 32), 0), (1, 1, (20480, 192), 1), (0, 1, (20480, 64), 1)])
def test_tiles_of_the_mxfp8_column_cast(lib, f32, blocked, size, narrow):
    assert lib.narrow_cols(f32, blocked, *size, CUS) == narrow
