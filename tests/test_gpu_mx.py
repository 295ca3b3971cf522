"""GPU parity: mx_fp8_quantize (all orientations and scale layouts) bit for bit against the CPU
oracle, and mx_fp8_bf16 against the dequantized matmul, on the reference's shape lists
(test/test_mx.py:42-59,70-84) and the benchmark configs."""
import pytest
import torch

from oracle import c_oracle as co
from oracle import eager
from tests import util
from tests.test_ring_plan import SHARES

pytestmark = pytest.mark.gpu

E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2


@pytest.fixture(scope="module")
def d(gpu_device):
    import driss_torch_amd

    return driss_torch_amd


@pytest.fixture(scope="module")
def cabi(gpu_device):
    from driss_torch_amd import cabi as c

    return c


# --------------------------------------------------------------------------- MX cast
@pytest.mark.parametrize("size", [(128, 32), (256, 32), (8192, 32), (128, 64), (128, 128), (128, 8192), (256, 64),
                                  (256, 128), (8192, 8192)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_mx_cast_reference_shapes(d, size):
    """test/test_mx.py:70-94: positive uniform bf16 input, data and scale bit exact"""
    a = util.uniform(size, 400 + size[0] + size[1])
    data, scale = d.mx_fp8_quantize(a.cuda())
    assert data.dtype == E4 and data.shape == a.shape
    assert scale.dtype == torch.float8_e8m0fnu and scale.shape == (size[0] * size[1] // 32,)
    rd, rs = co.mx_quantize(a)
    assert torch.equal(util.codes(scale), rs.flatten())
    assert torch.equal(util.codes(data), rd)
    if size[0] * size[1] <= 1 << 20:
        es, ed = eager.to_mx(a, E4)
        assert torch.equal(util.codes(scale), es.flatten()) and torch.equal(util.codes(data), util.codes(ed))


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("out_dtype", [E4, E5])
@pytest.mark.parametrize("axis,transpose", [(1, False), (0, False), (0, True), (1, True)])
@pytest.mark.parametrize("shape", [(32, 32), (96, 160), (160, 96), (512, 1056), (1056, 512)])
def test_mx_cast_orientations(d, in_dtype, out_dtype, axis, transpose, shape):
    a = util.student_t(shape, 500 + shape[0], in_dtype)
    a[0, 0] = 0.0
    a[-1, -1] = -0.0
    if in_dtype != torch.float16:
        a[3, 5] = 3e38 if in_dtype == torch.float32 else 3e38
    data, scale = d.mx_fp8_quantize(a.cuda(), 32, axis, transpose, out_dtype)
    rd, rs = co.mx_quantize(a, axis=axis, transpose=transpose, out_dtype=out_dtype)
    assert data.shape == rd.shape and scale.numel() == rs.numel()
    assert torch.equal(util.codes(scale), rs.flatten())
    assert torch.equal(util.codes(data), rd)


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("axis,transpose", [(1, False), (0, False), (0, True)])
def test_mx_cast_special_blocks(d, in_dtype, axis, transpose):
    a = util.student_t((64, 128), 61, in_dtype)
    a[0:32, 0:32] = 0                      # all-zero blocks in either direction -> byte 0, zero payload
    a[40, 70] = float("nan")               # NaN block -> byte 255, NaN payload
    a[33, 33] = float("inf")               # inf saturates, byte from exponent 128
    tiny = 1e-40 if in_dtype == torch.float32 else (2.0 ** -133 if in_dtype == torch.bfloat16 else 2.0 ** -24)
    a[32:64, 96:128] = tiny                # subnormal maxima
    a[:, 100] = torch.where(torch.arange(64) % 2 == 0, 1.0, -1.0).to(in_dtype) * tiny
    data, scale = d.mx_fp8_quantize(a.cuda(), 32, axis, transpose, E4)
    rd, rs = co.mx_quantize(a, axis=axis, transpose=transpose)
    assert torch.equal(util.codes(scale), rs.flatten())
    assert torch.equal(util.codes(data), rd)


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_mx_cast_input_off_a_16_byte_boundary(d, in_dtype):
    """a contiguous view that starts one element into its buffer: every orientation keeps its tiled
    kernel (the loads go through element-aligned vector types); all of them against the oracle"""
    rows, cols = 96, 544
    a = util.student_t((rows, cols), 61, in_dtype)
    buf = torch.empty(a.numel() + 3, dtype=in_dtype, device="cuda")
    buf[1:1 + a.numel()] = a.cuda().flatten()
    x = buf[1:1 + a.numel()].view(rows, cols)
    assert x.data_ptr() % 16 != 0
    rd, rs = co.mx_quantize(a, 1, False)
    data, scale = d.mx_fp8_quantize(x)
    assert torch.equal(util.codes(data), rd) and torch.equal(util.codes(scale), rs.flatten())
    data, scale = d.mx_fp8_quantize_blocked(x)
    assert torch.equal(util.codes(data), rd) and torch.equal(util.codes(scale), co.to_blocked(rs))
    cd, cs = co.mx_quantize(a, 0, True)
    data, scale = d.mx_fp8_quantize(x, 32, 0, True)
    assert torch.equal(util.codes(data), cd) and torch.equal(util.codes(scale), cs.flatten())
    dr, sr, dc, sc = d.mx_fp8_quantize_dual(x)
    assert torch.equal(util.codes(dr), rd) and torch.equal(util.codes(sr), rs.flatten())
    assert torch.equal(util.codes(dc), cd) and torch.equal(util.codes(sc), cs.flatten())
    for axis, transpose in ((0, False), (1, True)):
        wd, ws = co.mx_quantize(a, axis, transpose)
        data, scale = d.mx_fp8_quantize(x, 32, axis, transpose)
        assert torch.equal(util.codes(data), wd) and torch.equal(util.codes(scale), ws.flatten())


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(16, 32), (48, 96), (272, 544), (128, 8192), (4112, 256)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_mx_cast_rows_with_transposed_payload(d, in_dtype, shape):
    """(axis 1, transpose): the row-wise cast written as [cols, rows] with scales [cols/32, rows]; equal to the
    row-wise cast transposed, NaN and zero blocks included, on row counts that are multiples of 16 but not
    of 32 or 128, and through the general kernel when they are not multiples of 16"""
    a = util.student_t(shape, 901 + shape[0], in_dtype)
    a[0, :32] = 0
    a[shape[0] - 1, 5] = float("nan")
    rd, rs = co.mx_quantize(a, 1, False)
    data, scale = d.mx_fp8_quantize(a.cuda(), 32, 1, True)
    assert data.shape == (shape[1], shape[0])
    assert torch.equal(util.codes(data), rd.t()) and torch.equal(util.codes(scale).view(shape[1] // 32, shape[0]), rs.t())
    odd = a[:shape[0] - 3].contiguous() if shape[0] > 3 else a
    rd, rs = co.mx_quantize(odd, 1, False)
    data, scale = d.mx_fp8_quantize(odd.cuda(), 32, 1, True)
    assert torch.equal(util.codes(data), rd.t()) and torch.equal(util.codes(scale).view(shape[1] // 32, -1), rs.t())


def test_mx_cast_blocked_scales_and_errors(d, cabi):
    for shape, axis in [((256, 512), 1), ((129, 160), 1), ((512, 256), 0), ((160, 129 * 1), 0), ((96, 200), 0)]:
        a = util.student_t(shape, 71 + shape[0])
        data, scale = d.mx_fp8_quantize_blocked(a.cuda(), axis=axis)
        rd, rs = co.mx_quantize(a, axis=axis, transpose=(axis == 0))
        assert torch.equal(util.codes(data), rd)
        assert torch.equal(util.codes(scale), co.to_blocked(rs))
        # to_blocked on its own
        assert torch.equal(d.to_blocked(rs.cuda()).cpu(), eager.to_blocked(rs))
    x = util.student_t((64, 48), 72).cuda()
    with pytest.raises(RuntimeError):
        d.mx_fp8_quantize(x)  # 48 % 32 != 0 (src/mx_cast.cu:218-219)
    with pytest.raises(RuntimeError):
        d.mx_fp8_quantize(x.t())  # not contiguous
    with pytest.raises(RuntimeError):
        d.mx_fp8_quantize(x.double())
    with pytest.raises(RuntimeError):
        d.mx_fp8_quantize(x, 16)
    with pytest.raises(RuntimeError):
        d.mx_fp8_quantize(x, 32, 1, False, torch.bfloat16)
    assert d.mx_fp8_quantize(x, 32, 0)[0].shape == (64, 48)


def test_mx_cast_config4_full_size(d):
    a = util.student_t((8192, 8192), 1004)
    ag = a.cuda()
    data, scale = d.mx_fp8_quantize(ag)
    rd, rs = co.mx_quantize(a)
    assert torch.equal(util.codes(scale), rs.flatten()) and torch.equal(util.codes(data), rd)
    # column-wise blocks, output transposed == row-wise cast of x^T (checked against both)
    dT, sT = d.mx_fp8_quantize(ag, 32, 0, True)
    rdT, rsT = co.mx_quantize(a, axis=0, transpose=True)
    assert torch.equal(util.codes(sT), rsT.flatten()) and torch.equal(util.codes(dT), rdT)
    d2, s2 = d.mx_fp8_quantize(ag.t().contiguous())
    assert torch.equal(util.codes(d2), util.codes(dT)) and torch.equal(util.codes(s2), util.codes(sT))
    # column-wise blocks in place
    d0, s0 = d.mx_fp8_quantize(ag, 32, 0, False)
    assert torch.equal(util.codes(d0), rdT.t()) and torch.equal(util.codes(s0).view(256, 8192), rsT.t())
    # round trip: dequantized value within 2^-4 of the block maximum
    deq = eager.mx_dequant(data.cpu()[:256], rs[:256])
    x = a[:256].float().reshape(256, 256, 32)
    assert ((deq.reshape(256, 256, 32) - x).abs().amax(-1) <= x.abs().amax(-1) * 2**-4).all()


def test_mx_cast_transposed_columns_walked_tiles_ragged(d):
    """More tiles than the transposed column cast's grid of walking workgroups, with ragged last row and
    column tiles: every workgroup handles a second tile whose loads were in flight under its first."""
    a = util.student_t((2080, 8200), 1011)
    dT, sT = d.mx_fp8_quantize(a.cuda(), 32, 0, True)
    rdT, rsT = co.mx_quantize(a, axis=0, transpose=True)
    assert torch.equal(util.codes(sT), rsT.flatten()) and torch.equal(util.codes(dT), rdT)


# --------------------------------------------------------------------------- MX GEMM
def _operands(d, M, K, N, seed, dist="rand"):
    mk = util.uniform if dist == "rand" else util.normal
    a = mk((M, K), seed).cuda()
    b = mk((N, K), seed + 1).cuda()
    a_data, a_scale = d.mx_fp8_quantize(a)
    b_data, b_scale = d.mx_fp8_quantize(b)
    a_sc = a_scale.view(M, K // 32)
    b_sc = b_scale.view(N, K // 32)
    return a_data, a_sc, b_data, b_sc


def _check_gemm(d, M, K, N, seed, dist):
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, seed, dist)
    out = d.mx_fp8_bf16(a_data, b_data.t(), d.to_blocked(a_sc), d.to_blocked(b_sc))
    assert out.shape == (M, N) and out.dtype == torch.bfloat16
    ad, asc, bd, bsc = a_data.cpu(), util.codes(a_sc), b_data.cpu(), util.codes(b_sc)
    da, db = eager.mx_dequant(ad, asc), eager.mx_dequant(bd, bsc)
    ref = da.double() @ db.double().T
    got = out.cpu().double()
    sqnr = eager.compute_error(ref, got).item()
    # Tolerance.  The only rounding besides fp32 accumulation is the final bf16 store (relative
    # 2^-9); measured against sum_k |a||b| that bounds every entry, and gives an SQNR well
    # above 45 dB even for zero-mean data.  The reference's bar is SQNR > 80 dB against a
    # *bf16* matmul of the same operands on rand data (test/test_mx.py:64); against the exact
    # product a bf16 output cannot exceed ~57 dB, so the bar here is 50 dB plus the entrywise
    # bound.
    bound = da.abs().double() @ db.abs().double().T
    err = (got - ref).abs()
    assert (err <= bound * 2**-8 + 1e-30).all(), f"max rel {(err / bound).max().item():.3e}"
    assert sqnr > 50, sqnr
    return out, ref


@pytest.mark.parametrize("size", [(128, 128, 128), (256, 256, 256), (384, 384, 384), (512, 512, 512), (768, 768, 768),
                                  (1024, 1024, 1024), (128, 256, 384), (256, 384, 512), (129, 256, 384), (133, 512, 528)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
@pytest.mark.parametrize("dist", ["rand", "randn"])
def test_mx_gemm_reference_sizes(d, size, dist):
    M, K, N = size
    _check_gemm(d, M, K, N, 600 + M + N, dist)


@pytest.mark.parametrize("variant", [1, 2, 7])
@pytest.mark.parametrize("size", [(128, 128, 128), (512, 256, 640), (133, 512, 528), (300, 1024, 264)])
def test_mx_gemm_both_tile_shapes(d, cabi, variant, size):
    cabi.set_tuning("gemm.variant", variant)
    try:
        _check_gemm(d, *size, 700, "randn")
    finally:
        cabi.set_tuning("gemm.variant", 0)


@pytest.mark.parametrize("variant", [0, 1, 2, 5, 7])
@pytest.mark.parametrize("K", [32, 64, 96, 160, 224, 416, 1120])
def test_mx_gemm_k_of_any_whole_number_of_blocks(d, cabi, variant, K):
    """K a multiple of 32 but not of 128 (the reference's own scale-length check leaves multiples of 128
    only, src/mx_fp8_bf16.cu:197-205): the last step is partly filled, its missing K-blocks are the zero
    padding of the blocked scales, and the loads stay inside the rows.  The operands sit at the very end
    of their allocations and the rows past the matrix edge are poisoned with NaN codes, so a load that
    strays shows up as a NaN; the result is checked against the exact product."""
    cabi.set_tuning("gemm.variant", variant)
    try:
        _check_gemm(d, 133, K, 264, 1900 + K, "randn")
        # a contiguous operand: the byte after a row's K bytes is the next row's first -- poison a copy's
        # neighbours and compare
        a_data, a_sc, b_data, b_sc = _operands(d, 70, K, 136, 1950 + K, "randn")
        sa, sb = d.to_blocked(a_sc), d.to_blocked(b_sc)
        want = d.mx_fp8_bf16(a_data, b_data.t(), sa, sb)
        a_wide = torch.full((70, K + 128), 0x7F, dtype=torch.uint8, device="cuda")  # 0x7F = NaN
        b_wide = torch.full((136, K + 128), 0x7F, dtype=torch.uint8, device="cuda")
        a_wide[:, :K] = a_data.view(torch.uint8)
        b_wide[:, :K] = b_data.view(torch.uint8)
        got = d.mx_fp8_bf16(a_wide.view(E4)[:, :K], b_wide.view(E4)[:, :K].t(), sa, sb)
        assert torch.equal(got, want)
    finally:
        cabi.set_tuning("gemm.variant", 0)


def _poisoned_blocked(d, sc):
    """the blocked layout of scale matrix `sc` [R, C] with every padding byte (rows past R, K-blocks past C)
    set to 0xFF, the E8M0 NaN code, instead of zero"""
    R, C = sc.shape
    full = torch.full((-(-R // 128) * 128, -(-C // 4) * 4), 0xFF, dtype=torch.uint8, device=sc.device)
    full[:R, :C] = sc.view(torch.uint8)
    return d.to_blocked(full)


@pytest.mark.parametrize("variant", [0, 1, 2, 5, 7, 9])
@pytest.mark.parametrize("size", [(40, 96, 264), (133, 160, 264), (64, 1120, 520), (300, 416, 136), (16, 4128, 2048)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_ignores_the_padding_of_the_scale_buffers(d, cabi, variant, size):
    """the K-blocks past the end of K in a blocked scale buffer (K % 128 != 0) are padding that the caller may
    have left uninitialised: with every padding byte set to the NaN code the result is the same bits as with
    zeros, on every kernel (tiles of both sizes, shared K, few rows), for e4m3 and for e2m1 operands"""
    M, K, N = size
    if variant == 9 and M > 64:
        pytest.skip("the kernel for few rows takes at most 64")
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 4100 + K, "randn")
    cabi.set_tuning("gemm.variant", variant)
    try:
        want = d.mx_fp8_bf16(a_data, b_data.t(), d.to_blocked(a_sc), d.to_blocked(b_sc))
        got = d.mx_fp8_bf16(a_data, b_data.t(), _poisoned_blocked(d, a_sc), _poisoned_blocked(d, b_sc))
        assert not got.isnan().any() and torch.equal(got, want)
        # the same payload bytes read as e2m1 pairs: K/2 bytes hold K elements
        a4, b4 = a_data.view(torch.uint8)[:, :K // 2].contiguous(), b_data.view(torch.uint8)[:, :K // 2].contiguous()
        want4 = d.mx_fp4_bf16(a4, b4.t(), d.to_blocked(a_sc), d.to_blocked(b_sc))
        got4 = d.mx_fp4_bf16(a4, b4.t(), _poisoned_blocked(d, a_sc), _poisoned_blocked(d, b_sc))
        assert not got4.isnan().any() and torch.equal(got4, want4)
    finally:
        cabi.set_tuning("gemm.variant", 0)


@pytest.mark.parametrize("size", [(1, 640, 8), (16, 2048, 256), (17, 96, 2056), (33, 1120, 264), (48, 416, 136), (64, 8192, 512),
                                  (5, 32, 24), (64, 160, 16), (8, 416, 264), (9, 288, 40), (24, 1120, 136), (28, 416, 264),
                                  (40, 2048, 64), (52, 160, 520), (56, 2080, 72)], ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
@pytest.mark.parametrize("variant", [9, 10])
def test_mx_gemm_few_rows_kernel(d, cabi, size, variant):
    """the kernels for problems of at most 64 rows, the one that the rule takes (9) and the one with 16 columns per workgroup, K shared between its
    eight waves, B straight from memory (10): every count of 8-row halves of A's tiles, ragged M and N, K with a partly
    filled last 128-element step; forced here for every N, and checked against the exact product"""
    cabi.set_tuning("gemm.variant", variant)
    try:
        _check_gemm(d, *size, 2100 + size[0], "randn")
    finally:
        cabi.set_tuning("gemm.variant", 0)


@pytest.mark.parametrize("size", [(16, 256, 20008), (40, 416, 9008), (64, 128, 17000), (3, 1024, 33000)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
@pytest.mark.parametrize("knobs", [dict(tiles=0, steps=0, per_cu=0, stagger=1), dict(tiles=1, steps=1, per_cu=1, stagger=1),
                                   dict(tiles=2, steps=2, per_cu=1, stagger=0)], ids=lambda k: "-".join(f"{a}{b}" for a, b in k.items()))
def test_mx_gemm_few_rows_kernel_walks_many_column_groups(d, cabi, size, knobs):
    """more groups of columns than the grid has workgroups: a workgroup then takes several groups in turn, with
    the first batch of the next one already on its way while it adds up and stores the one in hand (the sums
    are parked in the LDS set that has just been used up); every launch shape, with and without the staggered
    walk along K; the exact product, and the same bits on a second call"""
    cabi.set_tuning("gemm.variant", 10)
    for k, v in knobs.items():
        cabi.set_tuning("gemm.few_rows_" + k, v)
    try:
        out, _ = _check_gemm(d, *size, 2500 + size[0], "randn")
        assert torch.equal(_check_gemm(d, *size, 2500 + size[0], "randn")[0], out)
    finally:
        cabi.set_tuning("gemm.variant", 0)
        for k, v in dict(tiles=0, steps=0, per_cu=0, stagger=1).items():
            cabi.set_tuning("gemm.few_rows_" + k, v)


def test_mx_gemm_few_rows_kernel_is_the_default_and_respects_strides(d, cabi):
    """with enough columns the library takes that kernel by itself; operands and output that are slices of
    wider tensors give the same bits, loads stay inside the rows (poisoned neighbours) and nothing is
    written outside the output"""
    M, K, N = 5, 4128, 4104
    out, _ = _check_gemm(d, M, K, N, 2200, "randn")
    cabi.set_tuning("gemm.variant", 9)
    try:
        a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 2200, "randn")
        sa, sb = d.to_blocked(a_sc), d.to_blocked(b_sc)
        assert torch.equal(d.mx_fp8_bf16(a_data, b_data.t(), sa, sb), out)
        a_wide = torch.full((M, K + 384), 0x7F, dtype=torch.uint8, device="cuda")  # 0x7F = NaN
        b_wide = torch.full((N, K + 640), 0x7F, dtype=torch.uint8, device="cuda")
        a_wide[:, 128:128 + K] = a_data.view(torch.uint8)
        b_wide[:, 256:256 + K] = b_data.view(torch.uint8)
        out_wide = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device="cuda")
        cabi.mx_fp8_bf16(a_wide.view(E4)[:, 128:128 + K], b_wide.view(E4)[:, 256:256 + K], sa, sb, out_wide[:, 8:8 + N])
        assert torch.equal(out_wide[:, 8:8 + N], out)
        assert (out_wide[:, :8] == 7.0).all() and (out_wide[:, 8 + N:] == 7.0).all()
    finally:
        cabi.set_tuning("gemm.variant", 0)


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("size", [(24, 2048, 8192), (16, 4096, 4096), (40, 4096, 4096), (24, 1312, 2048)], ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_split_k_leaves_the_few_rows_kernel_alone(d, cabi, size, fp4):
    """gemm.split_k says how the small tiles share K: a product that takes the kernel for few rows takes it under any factor (the order of
    its sums is its own, so the bits tell)"""
    M, K, N = size
    x, w = _wide_operand((M, K), 2700 + M).cuda(), _wide_operand((N, K), 2701).cuda()
    if fp4:
        (a, sa), (b, sb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
    else:
        (a, sa), (b, sb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
    outs = {}
    for variant, split_k in ((9, 0), (0, 0), (0, 1), (0, 3), (3, 1)):
        cabi.set_tuning("gemm.variant", variant)
        cabi.set_tuning("gemm.split_k", split_k)
        try:
            outs[variant, split_k] = op(a, b.t(), sa, sb)
        finally:
            cabi.set_tuning("gemm.variant", 0)
            cabi.set_tuning("gemm.split_k", 0)
    assert not torch.equal(outs[3, 1], outs[9, 0])
    for split_k in (0, 1, 3):
        assert torch.equal(outs[0, split_k], outs[9, 0]), split_k


def _random_gemm_sizes(seed, n):
    import random

    rng = random.Random(seed)
    return [(rng.randint(1, 700), 128 * rng.randint(1, 9), 8 * rng.randint(1, 100)) for _ in range(n)]


@pytest.mark.parametrize("variant", [0, 2, 5, 7])
@pytest.mark.parametrize("size", _random_gemm_sizes(7, 8), ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_random_sizes(d, cabi, variant, size):
    """(M, K, N) with M arbitrary, N a multiple of 8 (src/mx_fp8_bf16.cu:187), K a multiple of 128: ragged edge
    tiles in both directions"""
    cabi.set_tuning("gemm.variant", variant)
    try:
        _check_gemm(d, *size, 900 + size[0], "randn")
    finally:
        cabi.set_tuning("gemm.variant", 0)


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("K", [32, 96, 128, 160, 256, 288, 384, 512, 640, 672, 1024, 1184])
def test_mx_gemm_schedules_agree(d, cabi, fp4, K):
    """The schedule that holds a B fragment for all of A (256 x 256 and 256 x 192 tiles) against the quadrant
    one: every entry is summed in the same order, so the bits are the same.  One step, odd and even numbers of
    them, partly filled last steps, tiles that start in the middle of a chunk of scales, ragged edges."""
    M, N = 520, 776  # 192-column tiles at columns 192 (in the middle of a chunk) and 768 (8 columns in it)
    x, w = _wide_operand((M, K), 3000 + K).cuda(), _wide_operand((N, K), 3001 + K).cuda()
    if fp4:
        (a, sa), (b, sb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
    else:
        (a, sa), (b, sb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
    outs = {}
    for variant in (7, 2, 5):
        cabi.set_tuning("gemm.variant", variant)
        try:
            outs[variant] = op(a, b.t(), sa, sb)
        finally:
            cabi.set_tuning("gemm.variant", 0)
    assert torch.isfinite(outs[7]).all() and outs[7].abs().max() > 0
    assert torch.equal(outs[2], outs[7]) and torch.equal(outs[5], outs[7])


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("K", [96, 160, 256, 384, 672, 768, 1120, 1280, 1312])
def test_mx_gemm_schedules_agree_on_every_form_of_operand(d, cabi, fp4, K):
    """The same comparison, and the small tiles beside it, on what a caller may pass beside library-made contiguous operands: padding of the scales
    full of NaN codes, row strides above K, an output inside a wider one that begins 8 bytes off a 16-byte boundary,
    a row count and a column count that are no multiples of 8 -- for every number of steps, odd and even, whole and
    partly filled last ones."""
    M, N = 300, 580  # four tiles of 192 columns, the last with 4
    kb = K // 2 if fp4 else K
    x, w = _wide_operand((M, K), 4000 + K).cuda(), _wide_operand((N, K), 4001 + K).cuda()
    quantize = cabi.mx_fp4_quantize if fp4 else cabi.mx_fp8_quantize
    product = cabi.mx_fp4_bf16 if fp4 else cabi.mx_fp8_bf16
    (a, sa), (b, sb) = ((q.view(torch.uint8), s.view(torch.uint8).view(-1, K // 32)) for q, s in (quantize(x), quantize(w)))
    dtype = torch.uint8 if fp4 else E4

    def strided(t, before, after):
        wide = torch.full((t.shape[0], before + kb + after), 0x7F, dtype=torch.uint8, device="cuda")
        wide[:, before:before + kb] = t
        return wide[:, before:before + kb].view(dtype)

    a_view, b_view = strided(a, 16, 48 - kb % 16), strided(b, 64, 16 - kb % 16)
    outs = {}
    small = [(3, tm, tn) for tm in (64, 128) for tn in (64, 128)]
    for variant in [7, 2, 5] + small:
        number, tm, tn = variant if variant in small else (variant, 0, 0)
        knobs = {"gemm.variant": number, "gemm.tile_m": tm, "gemm.tile_n": tn, "gemm.split_k": 1 if tm else 0}
        for k, v in knobs.items():
            cabi.set_tuning(k, v)
        try:
            outs[variant] = product(a.view(dtype), b.view(dtype), d.to_blocked(sa), d.to_blocked(sb))
            for lead, pitch in ((4, N + 24), (8, N + 28)):  # 8 bytes off a boundary; on it, with a pitch of whole vectors
                out = torch.full((M, pitch), 7.0, dtype=torch.bfloat16, device="cuda")
                product(a_view, b_view, _poisoned_blocked(d, sa), _poisoned_blocked(d, sb), out[:, lead:lead + N])
                assert torch.equal(out[:, lead:lead + N], outs[variant]), (variant, lead)
                assert (out[:, :lead] == 7.0).all() and (out[:, lead + N:] == 7.0).all(), (variant, lead)
        finally:
            for k in knobs:
                cabi.set_tuning(k, 0)
    assert torch.isfinite(outs[7]).all() and outs[7].abs().max() > 0
    assert all(torch.equal(out, outs[7]) for out in outs.values())


def _wide_operand(shape, seed):
    """N(0, 1) rows with scales that differ from block to block, so that a scale of the wrong row or block shows"""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g).view(shape[0], -1, 32)
    return (x * torch.exp2(torch.randint(-6, 7, x.shape[:2] + (1,), generator=g).float())).view(shape).bfloat16()


@pytest.mark.parametrize("splits", [0, 2, 3, 5, 16])
@pytest.mark.parametrize("size", [(16, 2048, 256), (133, 1664, 264), (300, 1024, 136), (1, 640, 8), (64, 8192, 512),
                                  (40, 4192, 136)], ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_split_k(d, cabi, splits, size):
    """K shared between several workgroups per tile (forced factors, and the library's own choice):
    same tolerance as the plain kernel, the same bits on every call (the sum runs in split order
    whoever finishes last, and the ticket counters come back to zero), uneven shares of K-steps."""
    cabi.set_tuning("gemm.split_k", splits)
    try:
        out, _ = _check_gemm(d, *size, 1100 + size[0], "randn")
        for _ in range(3):
            again, _ = _check_gemm(d, *size, 1100 + size[0], "randn")
            assert torch.equal(again, out)
    finally:
        cabi.set_tuning("gemm.split_k", 0)


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("size", SHARES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_few_shares_by_rule(d, cabi, size, fp4):
    """Products whose K the library's own rule shares, evenly and not, and some that it does not (how many shares each has is checked
    where the rule is): integers of at most 4 times a power of two of each block's own, up to 2^3 in one operand and 2^2 in
    the other, so that a share that took its scales elsewhere along K would show, and every partial sum
    (at most 2^9 K < 2^24) is exact in fp32 whatever the order: the result is one bit pattern."""
    M, K, N = size
    g = torch.Generator(device="cuda").manual_seed(M + K)

    def integers(rows, top):
        v = torch.randint(-4, 5, (rows, K // 32, 32), generator=g, device="cuda").float()
        return (v * torch.exp2(torch.randint(0, top + 1, (rows, K // 32, 1), generator=g, device="cuda").float())).view(rows, K)

    a, b = integers(M, 3), integers(N, 2)
    want = (a @ b.t()).bfloat16()
    if fp4:
        (qa, sa), (qb, sb) = (d.mx_fp4_quantize(t.bfloat16(), blocked=True) for t in (a, b))
        product = d.mx_fp4_bf16
    else:
        (qa, sa), (qb, sb) = (d.mx_fp8_quantize_blocked(t.bfloat16()) for t in (a, b))
        product = d.mx_fp8_bf16
    for _ in range(2):  # the second call finds the tickets as the first one left them
        assert torch.equal(product(qa, qb.t(), sa, sb), want)


@pytest.mark.parametrize("size", [(4352, 256, 4096), (4100, 256, 4360), (4352, 384, 4352), (8200, 128, 4104),
                                  (2304, 128, 2304), (2200, 256, 2312)],  # the last two: 81 and 90 tiles, halves only
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_leftover_tiles_as_quadrants(d, cabi, size):
    """more 256 x 256 tiles than CUs: whole rounds on the big kernel, the tiles left over as 128 x 128
    quadrants or 256 x 128 halves (forced here, whatever the library would pick): every entry written once and right, with
    tile counts that are and are not multiples of 8 and ragged edges in both directions"""
    outs = []
    for tail in (0, 2, 3):  # the big kernel alone, leftover as quadrants, leftover as 256 x 128 halves
        cabi.set_tuning("gemm.tail_quads", tail)
        try:
            outs.append(_check_gemm(d, *size, 1400 + size[0], "randn")[0])
        finally:
            cabi.set_tuning("gemm.tail_quads", 1)
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])  # same K order per entry: the same bits


@pytest.mark.parametrize("size", [(300, 1024, 264), (64, 8192, 512), (2304, 256, 2304), (4100, 256, 4360)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_strided_operands_and_output(d, cabi, size):
    """operands that are column slices of wider matrices (row stride > K, data pointer off the
    allocation's start) and an output that is a slice of a wider one: the same bits as with
    contiguous tensors, on every launch plan"""
    M, K, N = size
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 1600 + M, "randn")
    sa, sb = d.to_blocked(a_sc), d.to_blocked(b_sc)
    want = d.mx_fp8_bf16(a_data, b_data.t(), sa, sb)
    a_wide = torch.zeros((M, K + 384), dtype=torch.uint8, device="cuda").view(E4)
    b_wide = torch.zeros((N, K + 640), dtype=torch.uint8, device="cuda").view(E4)
    a_wide[:, 128:128 + K] = a_data
    b_wide[:, 256:256 + K] = b_data
    a_view, b_view = a_wide[:, 128:128 + K], b_wide[:, 256:256 + K]
    assert a_view.stride(0) == K + 384 and not a_view.is_contiguous()
    assert torch.equal(d.mx_fp8_bf16(a_view, b_view.t(), sa, sb), want)
    out_wide = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device="cuda")
    cabi.mx_fp8_bf16(a_view, b_view, sa, sb, out_wide[:, 8:8 + N])
    assert torch.equal(out_wide[:, 8:8 + N], want)
    assert (out_wide[:, :8] == 7.0).all() and (out_wide[:, 8 + N:] == 7.0).all()  # nothing written outside


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("size", [(128, 288, 32512), (65, 288, 32520), (128, 256, 32768), (128, 288, 32776), (32700, 256, 128)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_one_band_of_rows(d, cabi, size, fp4):
    """A band of at most 128 rows (or columns) around the width where its 128 x 128 tiles are one round of the
    chip and its 256 x 256 tiles half of one: the same bits as on 128 x 128 tiles, whatever is picked."""
    M, K, N = size
    x, w = _wide_operand((M, K), 5000 + M).cuda(), _wide_operand((N, K), 5001 + N).cuda()
    if fp4:
        (a, sa), (b, sb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
    else:
        (a, sa), (b, sb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
    got = op(a, b.t(), sa, sb)
    cabi.set_tuning("gemm.variant", 1)
    try:
        assert torch.equal(op(a, b.t(), sa, sb), got)
    finally:
        cabi.set_tuning("gemm.variant", 0)
    assert torch.isfinite(got).all() and got.abs().max() > 0


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("tile", [(64, 64), (64, 128), (128, 64), (128, 128)], ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("size", [(1, 32, 8), (64, 128, 64), (129, 96, 72), (65, 544, 136),  # one step, one line of a row in part
                                  (128, 512, 128), (100, 640, 200), (130, 1024, 264), (60, 1056, 520),  # as many steps as stages, one more
                                  (192, 2048, 192), (33, 2080, 264), (257, 2272, 328), (400, 2560, 72)],  # every stage more than once
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_small_tiles(d, cabi, size, tile, fp4):
    """The kernel for few tiles, every tile of it forced: the same K order per entry as the 256 x 256 tiles have, so the same
    bits; with rows that are whole lines and with rows off them (contiguous, and as slices that begin 16 and 48 bytes into a line,
    their neighbours poisoned); and shares of K within fp32 rounding of the sums."""
    M, K, N = size
    x, w = _wide_operand((M, K), 7000 + M).cuda(), _wide_operand((N, K), 7001 + N).cuda()
    if fp4:
        (a, sa), (b, sb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
    else:
        (a, sa), (b, sb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
    knobs = {"gemm.variant": 2, "gemm.tile_m": tile[0], "gemm.tile_n": tile[1], "gemm.split_k": 1}
    try:
        for k, v in knobs.items():
            cabi.set_tuning(k, v)
        want = op(a, b.t(), sa, sb)
        assert torch.isfinite(want).all() and want.abs().max() > 0
        # shares of K, the sum in another order: an MFMA keeps 2^-22 of its largest addend, an addition of two sums 2^-24, at most 20 of
        # each here: 2^-17 of the sum of magnitudes; then one bf16 rounding (8 significant bits: 2^-8 at most) on either side
        bound = 2.0 ** -7 * want.float().abs() + 2.0 ** -17 * _abs_product(op, a, b, sa, sb)
        cabi.set_tuning("gemm.variant", 3)
        kb = a.shape[1]
        for _ in range(2):
            assert torch.equal(op(a, b.t(), sa, sb), want)

        def inside(t, lead, pitch):  # as columns of a wider matrix of NaN codes
            wide = torch.full((t.shape[0], pitch), 0x7F, dtype=torch.uint8, device="cuda")
            wide[:, lead:lead + kb] = t.view(torch.uint8)
            return wide.view(t.dtype)[:, lead:lead + kb]

        for lead_a, lead_b in ((16, 48), (0, 112)):
            pitch = -(-(kb + 128) // 16) * 16 + 16 * (lead_b // 48)
            assert torch.equal(op(inside(a, lead_a, pitch), inside(b, lead_b, pitch + 32).t(), sa, sb), want)
        for splits in (2, 3, 5):
            cabi.set_tuning("gemm.split_k", splits)
            got = op(a, b.t(), sa, sb)
            assert ((got.float() - want.float()).abs() <= bound).all()
            assert torch.equal(op(a, b.t(), sa, sb), got)
    finally:
        for k in knobs:
            cabi.set_tuning(k, 0)


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("size", [(512, 4096, 4096), (487, 3840, 3728), (390, 8192, 264), (300, 7168, 1024), (1000, 2080, 2048), (64, 4096, 1024)],
                         ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_equal_rows_have_equal_results(d, cabi, size, fp4):
    """A row's result does not depend on where in `a` it stands, on any plan: with one row for all of `a`, all rows of the product are the
    same bits, and so are all columns with one row for all of `b`."""
    M, K, N = size
    quantize, op = (d.mx_fp4_quantize, d.mx_fp4_bf16) if fp4 else (d.mx_fp8_quantize_blocked, d.mx_fp8_bf16)
    quantized = lambda x: quantize(x.cuda(), blocked=True) if fp4 else quantize(x.cuda())  # noqa: E731
    x, w = _wide_operand((M, K), 7300 + M), _wide_operand((N, K), 7301)
    (a, sa), (b, sb) = quantized(x), quantized(w)
    (a1, sa1), (b1, sb1) = quantized(x[:1].expand(M, K).contiguous()), quantized(w[:1].expand(N, K).contiguous())
    got = op(a1, b.t(), sa1, sb)
    assert got.abs().max() > 0 and torch.equal(got, got[:1].expand(M, N))
    got = op(a, b1.t(), sa, sb1)
    assert got.abs().max() > 0 and torch.equal(got, got[:, :1].expand(M, N))


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("rows", [384, 385])
@pytest.mark.parametrize("steps", [15, 16, 17])
def test_mx_gemm_rows_off_the_lines_on_halves_or_small_tiles(d, cabi, rows, steps, fp4):
    """either side of the lines between the two (which size takes which is checked where the rule is), the last step a quarter full: the
    same K order, so the bits of the 256 x 256 tiles"""
    K, N = ((steps - 1) * 128 + 32) * (2 if fp4 else 1), 12008
    x, w = _wide_operand((rows, K), 7100 + steps).cuda(), _wide_operand((N, K), 7101).cuda()
    if fp4:
        (a, sa), (b, sb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
    else:
        (a, sa), (b, sb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
    got = op(a, b.t(), sa, sb)
    cabi.set_tuning("gemm.variant", 2)
    try:
        assert torch.equal(op(a, b.t(), sa, sb), got)
    finally:
        cabi.set_tuning("gemm.variant", 0)
    assert torch.isfinite(got).all() and got.abs().max() > 0


def _abs_product(op, a, b, sa, sb):
    """sum over k of |a| |b| with the signs of the codes taken off"""
    def magnitude(t):
        return (t.view(torch.uint8) & (0x7F if t.dtype == E4 else 0x77)).view(t.dtype)

    return op(magnitude(a), magnitude(b).t(), sa, sb).float() * (1 + 2.0 ** -7)


def _random_plan_sizes(seed, n):
    import random

    rng = random.Random(seed)
    return [(rng.randint(1, 6000), 128 * rng.randint(1, 3), 8 * rng.randint(1, 750)) for _ in range(n)]


@pytest.mark.parametrize("size", _random_plan_sizes(11, 10), ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_mx_gemm_random_sizes_across_launch_plans(d, size):
    """random (M, K, N) up to 6000 x 6000 outputs, ragged in both directions: whichever plan the
    library picks (small tiles, 256 x 128 tiles, whole rounds of big tiles with the leftover as
    quadrants or halves), every entry is within the tolerance of the fp32 product of the
    dequantized operands (computed on the device: a library matmul is the reference here)"""
    M, K, N = size
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    a = torch.randn((M, K), generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)
    b = torch.randn((N, K), generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)
    a_data, a_scale = d.mx_fp8_quantize(a)
    b_data, b_scale = d.mx_fp8_quantize(b)
    out = d.mx_fp8_bf16(a_data, b_data.t(), d.to_blocked(a_scale.view(M, K // 32)), d.to_blocked(b_scale.view(N, K // 32)))

    def dequant(data, scale, rows):
        s = torch.exp2(scale.view(torch.uint8).view(rows, K // 32).float() - 127.0).repeat_interleave(32, dim=1)
        return data.float() * s

    da, db = dequant(a_data, a_scale, M), dequant(b_data, b_scale, N)
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        ref = da @ db.T
        bound = da.abs() @ db.abs().T
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev
    err = (out.float() - ref).abs()
    assert bool((err <= bound * 2**-8 + 1e-30).all()), f"max rel {(err / bound).max().item():.3e}"


def test_mx_gemm_split_k_on_two_streams(d):
    """split-K products issued alternately on two streams (each stream has its own ticket counters and
    parking space in the torch shim): every result equals the one computed alone"""
    M, K, N = 48, 8192, 384
    ops = []
    for seed in (1700, 1710):
        a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, seed, "randn")
        ops.append((a_data, b_data.t(), d.to_blocked(a_sc), d.to_blocked(b_sc)))
    want = [d.mx_fp8_bf16(*o) for o in ops]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for rep in range(12):
        with torch.cuda.stream(streams[rep % 2]):
            got.append((rep % 2, d.mx_fp8_bf16(*ops[rep % 2])))
    torch.cuda.synchronize()
    for which, out in got:
        assert torch.equal(out, want[which])


def test_mx_gemm_split_k_workspace_rules(d, cabi):
    M, K, N = 32, 8192, 256  # 64 K-steps on 2 tiles: the library splits by itself
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 1200, "randn")
    sa, sb = d.to_blocked(a_sc), d.to_blocked(b_sc)
    with_ws = cabi.mx_fp8_bf16(a_data, b_data, sa, sb)
    without = cabi.mx_fp8_bf16(a_data, b_data, sa, sb, workspace=False)
    ref = eager.mx_dequant(a_data.cpu(), util.codes(a_sc)).double() @ eager.mx_dequant(b_data.cpu(), util.codes(b_sc)).double().T
    for got in (with_ws, without):
        assert eager.compute_error(ref, got.cpu().double()).item() > 50
    L = cabi.lib()
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ws = torch.full((L.dt_mx_gemm_workspace_bytes() + 256,), 0xAB, dtype=torch.uint8, device="cuda")
    assert L.dt_mx_gemm_workspace_init(ws.data_ptr(), ws.numel(), None) == 0  # zeroes the ticket counters
    args = (a_data.data_ptr(), b_data.data_ptr(), sa.data_ptr(), sb.data_ptr(), M, N, K, K, K, out.data_ptr(), N)
    assert L.dt_mx_fp8_bf16_ws(*args, ws.data_ptr() + 8, ws.numel() - 8, None) == 4  # misaligned workspace
    # a workspace too small for any split: the product is computed without one
    assert L.dt_mx_fp8_bf16_ws(*args, ws.data_ptr(), 1024, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, without)
    assert L.dt_mx_fp8_bf16_ws(*args, ws.data_ptr(), ws.numel() - 256, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, with_ws)
    assert int(ws[:1024].view(torch.int32).abs().sum().item()) == 0  # tickets are back at zero


def test_mx_gemm_small_vs_c_oracle_exact_products(d):
    """with power-of-two operands in a narrow exponent range every product and partial sum is
    exact, so the bf16 result must equal the C oracle's float64 reference rounded to bf16, bit
    for bit.  (Over a 2^22 range the MFMA's internal alignment drops the smallest addends --
    measured: 2 of 21760 entries lose a 2^-12 term next to 2^10 ones -- hence the range here.)"""
    M, K, N = 160, 256, 136
    g = util.gen(81)
    a = torch.exp2(torch.randint(-3, 3, (M, K), generator=g).float()) * torch.where(torch.rand(M, K, generator=g) < 0.5, -1.0, 1.0)
    b = torch.exp2(torch.randint(-3, 3, (N, K), generator=g).float()) * torch.where(torch.rand(N, K, generator=g) < 0.5, -1.0, 1.0)
    # sparse so that sums stay within bf16's 8 significant bits
    a = a * (torch.rand(M, K, generator=g) < 0.02)
    b = b * (torch.rand(N, K, generator=g) < 0.5)
    ad, asc = d.mx_fp8_quantize(a.bfloat16().cuda())
    bd, bsc = d.mx_fp8_quantize(b.bfloat16().cuda())
    out = d.mx_fp8_bf16(ad, bd.t(), d.to_blocked(asc.view(M, K // 32)), d.to_blocked(bsc.view(N, K // 32)))
    ref = co.mx_gemm_ref(util.codes(ad), util.codes(bd), co.to_blocked(util.codes(asc).view(M, K // 32)),
                         co.to_blocked(util.codes(bsc).view(N, K // 32)))
    assert torch.equal(out.cpu(), ref.bfloat16())


@pytest.mark.parametrize("size", [(16, 256, 136), (40, 352, 264), (64, 1152, 48)], ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("variant", [9, 10])
def test_mx_gemm_few_rows_kernel_vs_c_oracle_exact_products(d, cabi, size, tiles, variant):
    """the kernels for few rows on operands whose products and partial sums are exact (see the test above):
    bit for bit the C oracle's float64 reference rounded to bf16, for one and two 16-column tiles per
    wave and a K with a partly filled last step"""
    M, K, N = size
    g = util.gen(84 + M)
    a = torch.exp2(torch.randint(-3, 3, (M, K), generator=g).float()) * torch.where(torch.rand(M, K, generator=g) < 0.5, -1.0, 1.0)
    b = torch.exp2(torch.randint(-3, 3, (N, K), generator=g).float()) * torch.where(torch.rand(N, K, generator=g) < 0.5, -1.0, 1.0)
    a = a * (torch.rand(M, K, generator=g) < 0.02)
    b = b * (torch.rand(N, K, generator=g) < 0.5)
    ad, asc = d.mx_fp8_quantize(a.bfloat16().cuda())
    bd, bsc = d.mx_fp8_quantize(b.bfloat16().cuda())
    cabi.set_tuning("gemm.variant", variant)
    cabi.set_tuning("gemm.few_rows_tiles", tiles)
    try:
        out = d.mx_fp8_bf16(ad, bd.t(), d.to_blocked(asc.view(M, K // 32)), d.to_blocked(bsc.view(N, K // 32)))
    finally:
        cabi.set_tuning("gemm.variant", 0)
        cabi.set_tuning("gemm.few_rows_tiles", 0)
    ref = co.mx_gemm_ref(util.codes(ad), util.codes(bd), co.to_blocked(util.codes(asc).view(M, K // 32)),
                         co.to_blocked(util.codes(bsc).view(N, K // 32)))
    assert torch.equal(out.cpu(), ref.bfloat16())


def test_mx_gemm_scale_bytes_are_applied_per_row_and_kblock(d):
    M, K, N = 256, 512, 256
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 83, "randn")
    base = d.mx_fp8_bf16(a_data, b_data.t(), d.to_blocked(a_sc), d.to_blocked(b_sc)).float()
    sc2 = util.codes(a_sc).clone()
    sc2[77, :] += 3  # scale row 77 of A by 8
    out = d.mx_fp8_bf16(a_data, b_data.t(), d.to_blocked(sc2.cuda()), d.to_blocked(b_sc)).float()
    assert torch.equal(out[77], base[77] * 8)
    assert torch.equal(out[:77], base[:77]) and torch.equal(out[78:], base[78:])
    # zero all but one K-block of B: result equals the partial product of that block
    kb = 5
    b2 = util.codes(b_data).clone()
    mask = torch.zeros(K, dtype=torch.bool)
    mask[kb * 32:(kb + 1) * 32] = True
    b2[:, ~mask] = 0
    out = d.mx_fp8_bf16(a_data, b2.view(torch.float8_e4m3fn).cuda().t(), d.to_blocked(a_sc), d.to_blocked(b_sc))
    da = eager.mx_dequant(a_data.cpu(), util.codes(a_sc))[:, mask]
    db = eager.mx_dequant(b_data.cpu(), util.codes(b_sc))[:, mask]
    ref = (da.double() @ db.double().T)
    bound = da.abs().double() @ db.abs().double().T
    assert ((out.cpu().double() - ref).abs() <= bound * 2**-8).all()


def test_mx_gemm_argument_errors(d):
    M, K, N = 128, 128, 128
    a_data, a_sc, b_data, b_sc = _operands(d, M, K, N, 85)
    sa, sb = d.to_blocked(a_sc), d.to_blocked(b_sc)
    with pytest.raises(RuntimeError):
        d.mx_fp8_bf16(a_data, b_data, sa, sb)  # b not K-contiguous (src/mx_fp8_bf16.cu:211-213)
    with pytest.raises(RuntimeError):
        d.mx_fp8_bf16(a_data, b_data.t(), sa[:-1], sb)  # scale length (src/mx_fp8_bf16.cu:197-205)
    with pytest.raises(RuntimeError):
        d.mx_fp8_bf16(a_data[:, :64], b_data.t(), sa, sb)  # K mismatch
    with pytest.raises(RuntimeError):
        d.mx_fp8_bf16(a_data.view(torch.uint8), b_data.t(), sa, sb)
    with pytest.raises(RuntimeError):
        d.mx_fp4_bf16(a_data, b_data.t(), sa, sb)


def test_mx_gemm_config5_full_size(d):
    """8192^3 from the row-wise cast of N(0,1) operands, scales written blocked by the cast itself
    (1024 tiles of 256 x 256: four whole rounds of the chip).  Every entry of the output against the
    fp32 product of the dequantized operands, computed on the device (a library matmul is the
    reference), and sampled rows against the float64 product on the host."""
    M = N = K = 8192
    a = util.normal((M, K), 1005).cuda()
    b = util.normal((N, K), 1006).cuda()
    a_data, sa = d.mx_fp8_quantize_blocked(a)
    b_data, sb = d.mx_fp8_quantize_blocked(b)
    out = d.mx_fp8_bf16(a_data, b_data.t(), sa, sb)
    _, a_plain = d.mx_fp8_quantize(a)
    _, b_plain = d.mx_fp8_quantize(b)
    del a, b

    def dequant(data, scale, rows):
        s = torch.exp2(scale.view(torch.uint8).view(rows, K // 32).float() - 127.0).repeat_interleave(32, dim=1)
        return data.float() * s

    dga, dgb = dequant(a_data, a_plain, M), dequant(b_data, b_plain, N)
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        ref32 = dga @ dgb.T
        bound32 = dga.abs() @ dgb.abs().T
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev
    del dga, dgb
    err = (out.float() - ref32).abs()
    assert bool((err <= bound32 * 2**-8 + 1e-30).all()), f"max rel {(err / bound32).max().item():.3e}"
    sqnr_all = 20 * torch.log10(torch.norm(ref32) / torch.norm(out.float() - ref32))
    assert sqnr_all.item() > 50, sqnr_all.item()
    del err, ref32, bound32
    rows = torch.tensor([0, 1, 127, 128, 4095, 4096, 5000, 8191])
    da = eager.mx_dequant(a_data[rows.cuda()].cpu(), util.codes(a_plain).view(M, K // 32)[rows])
    db = eager.mx_dequant(b_data.cpu(), util.codes(b_plain).view(N, K // 32))
    ref = da.double() @ db.double().T
    got = out[rows.cuda()].cpu().double()
    bound = da.abs().double() @ db.abs().double().T
    assert ((got - ref).abs() <= bound * 2**-8).all()
    assert eager.compute_error(ref, got).item() > 50


@pytest.mark.parametrize("fp4", [False, True], ids=["e4m3", "e2m1"])
@pytest.mark.parametrize("octets", range(1, 9))
def test_mx_gemm_few_lines_kernel(d, cabi, octets, fp4):
    """the kernel for at most 32 rows by whole lines, every form of it: every number of column octets per group, and for every count of row octets fewer
    steps than waves and more than the stages of all of them, rows on the lines and off them; one step, columns that end inside an octet's chunk,
    several groups per workgroup; against the float64 product of the dequantized operands (bound per entry: bf16's rounding, 2^-8 of sum |a||b|), equal
    rows of A equal, and the same bits on a second call"""
    line = 256 if fp4 else 128
    every_form = [(M, K, 8 * octets + 136) for M in (2, 12, 20, 30) for steps in (3, 41) for K in (steps * line, steps * line + 32)]
    cabi.set_tuning("gemm.variant", 9)
    cabi.set_tuning("gemm.few_rows_octets", octets)
    try:
        for M, K, N in ((1, 32, 8), (8, 128, 8 * octets), (9, 1024, 136), (16, 2048, 264), (17, 1056, 1000), (25, 4160, 72), (32, 8192, 512),
                        (31, 96, 128 * octets + 8), (32, 256, 2048 * octets + 136), (3, 288, 4096 * octets + 40), *every_form):
            x, w = _wide_operand((M, K), 5000 + M + octets).cuda(), _wide_operand((N, K), 5001 + K).cuda()
            x[M - 1] = x[0]
            if fp4:
                (a, ba), (b, bb), op = d.mx_fp4_quantize(x, True), d.mx_fp4_quantize(w, True), d.mx_fp4_bf16
                a_val, b_val = (co.fp4_unpack(v).double() * torch.exp2(s.double() - 127).repeat_interleave(32, dim=1)
                                for v, s in (co.mx_fp4_quantize(t.cpu()) for t in (x, w)))
            else:
                (a, ba), (b, bb), op = d.mx_fp8_quantize_blocked(x), d.mx_fp8_quantize_blocked(w), d.mx_fp8_bf16
                a_val, b_val = (co.mx_dequant(*co.mx_quantize(t.cpu())).double() for t in (x, w))
            y = op(a, b.t(), ba, bb)
            exact, bound = a_val @ b_val.T, a_val.abs() @ b_val.abs().T
            assert ((y.cpu().double() - exact).abs() <= bound * 2**-8).all(), (M, K, N)
            assert torch.equal(y[M - 1], y[0]) and torch.equal(op(a, b.t(), ba, bb), y), (M, K, N)
    finally:
        cabi.set_tuning("gemm.variant", 0)
        cabi.set_tuning("gemm.few_rows_octets", 0)


@pytest.mark.parametrize("tile", [(64, 64), (64, 128), (128, 64), (128, 128)], ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("size", [(64, 8192, 1032), (200, 5120, 5120), (97, 8288, 1020), (300, 4192, 3004), (129, 4128, 2100), (257, 8256, 2760)],
                         ids=lambda s: "x".join(map(str, s)))
def test_mx_gemm_small_tiles_that_cover_fewer_columns(d, cabi, size, tile):
    """Tiles that begin anywhere in a chunk of B's scales, on and off whole lines, with columns that end inside a tile's eight: the same bits as on
    the 256 x 256 tiles (one order of sums), every entry within bf16's rounding of the float64 product, and nothing written past a row's end"""
    M, K, N = size
    x, w = _wide_operand((M, K), 6100 + M).cuda(), _wide_operand((N, K), 6101 + K).cuda()
    (a, sa), (b, sb) = ((q, _poisoned_blocked(d, s.view(torch.uint8).view(len(q), -1))) for q, s in (d.mx_fp8_quantize(x), d.mx_fp8_quantize(w)))
    a_val, b_val = (co.mx_dequant(*co.mx_quantize(t.cpu())).cuda().double() for t in (x, w))
    exact, bound = a_val @ b_val.T, a_val.abs() @ b_val.abs().T
    want = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    out = want.clone()
    for variant, dst in ((2, want), (3, out)):
        cabi.set_tuning("gemm.variant", variant)
        cabi.set_tuning("gemm.split_k", 1)
        cabi.set_tuning("gemm.tile_m", tile[0])
        cabi.set_tuning("gemm.tile_n", tile[1])
        try:
            cabi.mx_fp8_bf16(a, b, sa, sb, dst[:, :N])
        finally:
            for knob in ("variant", "split_k", "tile_m", "tile_n"):
                cabi.set_tuning("gemm." + knob, 0)
    assert torch.equal(out, want) and (out[:, N:] == 7).all()
    assert ((out[:, :N].double() - exact).abs() <= bound * 2**-8).all()
