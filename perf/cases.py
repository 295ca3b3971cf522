"""The calls that users of this package make, at the sizes they make them, as data and as code.

Six kinds of pass, each through the public wrappers of ``driss_torch``:

* ``delayed``  -- FP8 with delayed scaling: the amax of a tensor for the next step's scale, and its cast with
  the scale that the history gave for this one (``amax``, ``saturated_cast``).
* ``dynamic``  -- FP8 with a current per-tensor scale: ``dynamic_scaled_quant_ex`` (what
  ``dynamic_scaled_quant`` returns, with the amax and scale its consumer needs), or
  ``dynamic_scaled_quant_pair`` where a training step keeps an e4m3fn and an e5m2 copy.
* ``rowwise``  -- FP8 with one scale per token: ``dynamic_scaled_quant_rowwise``.
* ``mx_cast``  -- an MX operand made from a high-precision tensor: ``mx_fp8_quantize`` in the reference's form
  with row-major scales and ``to_blocked`` behind it, or ``mx_fp8_quantize_blocked`` along either axis.
* ``linear``   -- inference of one layer: the activations are quantized, the weights were when the model was
  loaded; 8 bits (``mx_fp8_quantize_blocked`` + ``mx_fp8_bf16``) or 4 (``mx_fp4_quantize`` + ``mx_fp4_bf16``).
  Few rows are decoding, many are prefill.
* ``train``    -- a training step of one layer: forward product and both gradients, with each of x, w and dy
  quantized along both of its axes from one read (``*_quantize_dual``).

Per-tensor dynamic quantization runs as a caller that does not own the GPU has it, i.e. without
``set_exclusive_gpu``.
"""
import math

import torch

import driss_torch as dt

E4, E5 = torch.float8_e4m3fn, torch.float8_e5m2
IN_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
OUT_DTYPES = {"e4m3fn": E4, "e5m2": E5}
IN_BYTES = {"bf16": 2, "f32": 4, "f16": 2}
FMAX = {"e4m3fn": 448.0, "e5m2": 57344.0}


def listed():
    return [
        # a small layer's tensor with delayed scaling: two short launches, latency is all there is
        {"name": "delayed_512x512", "kind": "delayed", "rows": 512, "cols": 512, "dtype": "bf16", "out": "e4m3fn"},
        # logits over a vocabulary, the widest tensor of the saturated-cast shape table
        {"name": "delayed_2048x109760", "kind": "delayed", "rows": 2048, "cols": 109760, "dtype": "bf16", "out": "e5m2"},
        # activations of one sequence of 1024 tokens: between latency and bandwidth
        {"name": "dynamic_1024x8192", "kind": "dynamic", "rows": 1024, "cols": 8192, "dtype": "bf16", "out": "e4m3fn"},
        # the benchmark's tensor: both FP8 copies of a training activation
        {"name": "dynamic_pair_8192x8192", "kind": "dynamic", "rows": 8192, "cols": 8192, "dtype": "bf16", "out": "pair"},
        # per-token scales of rows that are no whole number of 16-byte vectors
        {"name": "rowwise_8192x8190", "kind": "rowwise", "rows": 8192, "cols": 8190, "dtype": "bf16", "out": "e4m3fn"},
        # fp32 master weights turned into the operand of the weight-gradient side
        {"name": "mx_cast_cols_f32_3584x8192", "kind": "mx_cast", "rows": 3584, "cols": 8192, "dtype": "f32",
         "form": "blocked", "axis": 0},
        # decoding for a batch of 16 sequences
        {"name": "linear8_16x8192x8192", "kind": "linear", "bits": 8, "m": 16, "n": 8192, "k": 8192},
        # decoding for a large batch, or a short chunk of a prompt
        {"name": "linear8_200x14336x4096", "kind": "linear", "bits": 8, "m": 200, "n": 14336, "k": 4096},
        # prefill of a prompt of no round length
        {"name": "linear8_2000x5120x5120", "kind": "linear", "bits": 8, "m": 2000, "n": 5120, "k": 5120},
        # 4-bit weights, decoding
        {"name": "linear4_32x8192x8192", "kind": "linear", "bits": 4, "m": 32, "n": 8192, "k": 8192},
        # 4-bit weights, a long prefill
        {"name": "linear4_4096x8192x8192", "kind": "linear", "bits": 4, "m": 4096, "n": 8192, "k": 8192},
        # a training step of a wide layer, 8192 tokens
        {"name": "train8_8192x14336x4096", "kind": "train", "bits": 8, "m": 8192, "n": 14336, "k": 4096},
    ]


MOST_ELEMENTS = 2048 * 109760  # of a tensor to cast
MOST_MNK = 8192 * 14336 * 4096  # of the products of one training step, a third of its work


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, multiple=1):
    return max(lo, int(_log_uniform(rng, lo, hi)) // multiple * multiple)


def draw(rng):
    kind = rng.choice(["delayed", "dynamic", "rowwise", "mx_cast", "linear", "linear", "train"])
    if kind in ("delayed", "dynamic", "rowwise", "mx_cast"):
        total = _log_uniform(rng, 512 * 512, MOST_ELEMENTS)  # elements, then how they fall into rows
        multiple = 32 if kind == "mx_cast" else rng.choice([1, 1, 8, 128])
        cols = _size(rng, 512, 32768, multiple)
        rows = max(1, int(total / cols))
        if kind == "mx_cast":
            rows = max(32, rows // 32 * 32)
        case = {"kind": kind, "rows": rows, "cols": cols, "dtype": rng.choice(["bf16", "bf16", "f32"])}
        if kind == "mx_cast":
            case["dtype"] = rng.choice(["bf16", "bf16", "f32", "f16"])
            case["form"] = rng.choice(["plain", "blocked"])
            case["axis"] = 1 if case["form"] == "plain" else rng.choice([0, 1])
        else:
            case["out"] = rng.choice(["e4m3fn", "e5m2", "pair"] if kind == "dynamic" else ["e4m3fn", "e5m2"])
        return case
    bits = rng.choice([8, 8, 4])
    while True:
        if kind == "linear":
            m, n, k = _size(rng, 1, 8192), _size(rng, 1024, 28672, 8), _size(rng, 1024, 16384, 32)
        else:
            m, n, k = (_size(rng, 512, 14336, 32) for _ in range(3))
        if m * n * k <= MOST_MNK and n * k <= 16384 * 16384:
            return {"kind": kind, "bits": bits, "m": m, "n": n, "k": k}


# ------------------------------------------------------------------------------- inputs
def _normal(shape, gen, std=1.0, dtype=torch.bfloat16, outliers=0.0):
    """N(0, std) values; a share `outliers` of them a hundred times larger, as activations have them."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if std != 1.0:
        x.mul_(std)
    if outliers:
        n = max(1, int(x.numel() * outliers))
        at = torch.randint(0, x.numel(), (n,), generator=gen, device="cuda")
        x.view(-1)[at] *= 100.0
    return x.to(dtype)


def _inputs(case, seed):
    """The high-precision tensors of a case, on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": _normal((m, k), gen, outliers=1e-3), "w": _normal((n, k), gen, std=0.02)}
    if case["kind"] == "train":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": _normal((m, k), gen, outliers=1e-3), "w": _normal((n, k), gen, std=0.02),
                "dy": _normal((m, n), gen, std=1e-3)}
    shape, dtype = (case["rows"], case["cols"]), IN_DTYPES[case["dtype"]]
    if case["kind"] == "mx_cast":  # weights
        return {"x": _normal(shape, gen, std=0.02, dtype=dtype)}
    return {"x": _normal(shape, gen, dtype=dtype, outliers=1e-3)}


def _scale_of_history(x, out):
    """The 0-dim scale that delayed scaling has in hand: from an amax a little below this tensor's own."""
    return (FMAX[out] / (0.9 * x.abs().amax().double())).float()


def prepare(case, seed):
    state = {"case": case, **_inputs(case, seed)}
    if case["kind"] == "delayed":
        state["scale"] = _scale_of_history(state["x"], case["out"])
    elif case["kind"] == "linear":  # the weights of a loaded model: quantized once, the originals gone
        w = state.pop("w")
        quantize = dt.mx_fp8_quantize_blocked if case["bits"] == 8 else _fp4_blocked
        state["w_q"], state["w_s"] = quantize(w)
    return state


def _fp4_blocked(x):
    return dt.mx_fp4_quantize(x, blocked=True)


# -------------------------------------------------------------------------------- passes
def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


def _run_delayed(state, case):
    x = state["x"]
    return dt.amax(x), dt.saturated_cast(x, state["scale"], OUT_DTYPES[case["out"]])


def _run_dynamic(state, case):
    if case["out"] == "pair":
        return dt.dynamic_scaled_quant_pair(state["x"])
    return dt.dynamic_scaled_quant_ex(state["x"], OUT_DTYPES[case["out"]])


def _run_rowwise(state, case):
    return dt.dynamic_scaled_quant_rowwise(state["x"], OUT_DTYPES[case["out"]])


def _run_mx_cast(state, case):
    x = state["x"]
    if case["form"] == "plain":
        data, scale = dt.mx_fp8_quantize(x)
        scale = dt.to_blocked(scale.view(torch.uint8).view(x.shape[0], -1))
    else:
        data, scale = dt.mx_fp8_quantize_blocked(x, case["axis"])
        scale = scale.view(torch.uint8)
    return data, scale


def _run_linear(state, case):
    if case["bits"] == 8:
        x_q, x_s = dt.mx_fp8_quantize_blocked(state["x"])
        return dt.mx_fp8_bf16(x_q, state["w_q"].t(), x_s, state["w_s"])
    x_q, x_s = dt.mx_fp4_quantize(state["x"], blocked=True)
    return dt.mx_fp4_bf16(x_q, state["w_q"].t(), x_s, state["w_s"])


def _run_train(state, case):
    if case["bits"] == 8:
        def both(t):
            return dt.mx_fp8_quantize_dual(t, blocked=True)
        product = dt.mx_fp8_bf16
    else:
        def both(t):
            return dt.mx_fp4_quantize_dual(t, blocked=True)
        product = dt.mx_fp4_bf16
    x, x_s, x_t, x_ts = both(state["x"])
    w, w_s, w_t, w_ts = both(state["w"])
    y = product(x, w.t(), x_s, w_s)  # [M, N], along K
    dy, dy_s, dy_t, dy_ts = both(state["dy"])
    dx = product(dy, w_t.t(), dy_s, w_ts)  # [M, K], along N
    dw = product(dy_t, x_t.t(), dy_ts, x_ts)  # [N, K], along M
    return {"y": y, "dx": dx, "dw": dw}


_RUN = {"delayed": _run_delayed, "dynamic": _run_dynamic, "rowwise": _run_rowwise, "mx_cast": _run_mx_cast,
        "linear": _run_linear, "train": _run_train}


# ------------------------------------------------------------------------ what is needed
def work(case):
    if case["kind"] in ("linear", "train"):
        m, n, k = case["m"], case["n"], case["k"]
        if case["kind"] == "linear":
            w_bytes = n * k * case["bits"] // 8 + n * k // 32
            return {"bytes": 2 * m * k + w_bytes + 2 * m * n, "flops": 2 * m * n * k}
        return {"bytes": 2 * 2 * (m * k + n * k + m * n), "flops": 6 * m * n * k}
    n = case["rows"] * case["cols"]
    if case["kind"] == "mx_cast":
        return {"bytes": n * IN_BYTES[case["dtype"]] + n + n // 32, "flops": 0}
    copies = 2 if case["out"] == "pair" else 1
    per_row = 8 * case["rows"] if case["kind"] == "rowwise" else 0
    return {"bytes": n * (IN_BYTES[case["dtype"]] + copies) + per_row, "flops": 0}


def tolerance(case):
    if case["kind"] in ("linear", "train"):
        # fp32 sums of exact products, rounded to bf16: another order of summing moves a result across a rounding
        # boundary now and then (one unit in the last place, 2^-8 of the value at most)
        return {"rel": 2e-3, "max": 2e-2}
    return "exact"  # casts, maxima and scales have one answer


# ------------------------------------------------------------------ the same in 64 bits
def _blocks(x):
    return x.double().view(x.shape[0], -1, 32)


def _mx8(x):
    """(payload, scale) of the MXFP8 cast along the rows, before the payload is rounded: the scale is
    2^(ceil(log2 amax) - 8), float64."""
    b = _blocks(x)
    mant, exp = torch.frexp(b.abs().amax(-1, keepdim=True))  # amax = mant * 2^exp, mant in [0.5, 1)
    e = exp - (mant == 0.5).to(exp.dtype) - 8
    scale = torch.exp2(torch.where(mant == 0, -127, e.clamp(min=-127)).double())
    return (b / scale).clamp(-448.0, 448.0), scale


def _mx4(x):
    """The same for the MXFP4 cast: 2^(floor(log2 amax) - 2)."""
    b = _blocks(x)
    mant, exp = torch.frexp(b.abs().amax(-1, keepdim=True))
    scale = torch.exp2(torch.where(mant == 0, -127, (exp - 3).clamp(min=-127)).double())
    return b / scale, scale


def _as_quantized(x, bits):
    """What the quantized operand stands for, [rows, cols] in float64."""
    if bits == 8:
        v, scale = _mx8(x)
        v = v.float().to(E4).double()
    else:
        v, scale = _mx4(x)
        a = v.abs()
        step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0))  # the e2m1 grid: 0 .5 1 1.5 2 3 4 6
        v = torch.copysign((torch.round(a / step) * step).clamp(max=6.0), v)
    return (v * scale).view(x.shape)


def exact(case, seed):
    inputs = _inputs(case, seed)
    x = inputs["x"]
    if case["kind"] in ("linear", "train"):
        w, bits = inputs["w"], case["bits"]
        y = _as_quantized(x, bits) @ _as_quantized(w, bits).t()
        if case["kind"] == "linear":
            return y
        dy = inputs["dy"]
        dx = _as_quantized(dy, bits) @ _as_quantized(w.t().contiguous(), bits).t()
        dw = _as_quantized(dy.t().contiguous(), bits) @ _as_quantized(x.t().contiguous(), bits).t()
        return {"y": y, "dx": dx, "dw": dw}
    if case["kind"] == "mx_cast":
        if case["axis"] == 0:
            x = x.t().contiguous()
        return _mx8(x)[0].view(x.shape), None
    if case["kind"] == "delayed":
        scale = _scale_of_history(x, case["out"]).double()
        fmax = FMAX[case["out"]]
        return x.double().abs().amax().view(1), (x.double() * scale).clamp(-fmax, fmax)
    x = x.double()
    if case["kind"] == "rowwise":
        amax = x.abs().amax(-1, keepdim=True)
        scale = FMAX[case["out"]] / amax.clamp(min=1e-12)
        return x * scale, amax, scale
    amax = x.abs().amax()
    if case["out"] == "pair":
        scales = [FMAX["e4m3fn"] / amax.clamp(min=1e-12), FMAX["e5m2"] / amax.clamp(min=1e-12)]
        return x * scales[0], x * scales[1], amax.view(1), torch.stack(scales)
    scale = FMAX[case["out"]] / amax.clamp(min=1e-12)
    return x * scale, amax.view(1), scale
