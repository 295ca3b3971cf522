"""The wrappers as the tools that read a program take them: TorchScript compiles each of them, and torch.fx and function modes see the operator
that callers know, ``torch.ops.DrissTorch.<name>``."""
import inspect

import pytest
import torch
from torch.overrides import TorchFunctionMode

import driss_torch_amd as d

E4 = torch.float8_e4m3fn
PLAIN = torch.randn(32, 64)
# wrapper: the operator behind it, arguments
CALLS = {"amax": ("amax", (PLAIN,)),
         "saturated_cast": ("saturated_cast", (PLAIN, torch.ones(()), E4)),
         "saturated_cast_mode": ("saturated_cast_mode", (PLAIN, torch.ones(()), E4, 3)),
         "dynamic_scaled_quant": ("dynamic_scaled_quant", (PLAIN, E4)),
         "dynamic_scaled_quant_ex": ("dynamic_scaled_quant_ex", (PLAIN, E4)),
         "dynamic_scaled_quant_pair": ("dynamic_scaled_quant_pair", (PLAIN,)),
         "dynamic_scaled_quant_rowwise": ("dynamic_scaled_quant_rowwise", (PLAIN, E4)),
         "sweep_mm": ("sweep_mm", (PLAIN, PLAIN, PLAIN, PLAIN, None, torch.bfloat16, False, 1, 1, 1, False, 1)),
         "mx_fp8_bf16": ("mx_fp8_bf16", (PLAIN.to(E4), PLAIN.to(E4).t(), torch.zeros(512, dtype=torch.uint8), torch.zeros(512, dtype=torch.uint8))),
         "mx_fp4_bf16": ("mx_fp4_bf16", (torch.zeros(32, 32, dtype=torch.uint8), torch.zeros(32, 32, dtype=torch.uint8).t(),
                                         torch.zeros(512, dtype=torch.uint8), torch.zeros(512, dtype=torch.uint8))),
         "mx_fp8_quantize": ("mx_fp8_quantize", (PLAIN,)),
         "mx_fp8_quantize_blocked": ("mx_fp8_quantize_ex", (PLAIN,)),
         "mx_fp8_quantize_dual": ("mx_fp8_quantize_dual", (PLAIN,)),
         "mx_fp4_quantize": ("mx_fp4_quantize", (PLAIN,)),
         "mx_fp4_quantize_dual": ("mx_fp4_quantize_dual", (PLAIN,)),
         "to_blocked": ("to_blocked", (torch.zeros(32, 2, dtype=torch.uint8),))}


def test_every_wrapper_is_here():
    wrappers = {n for n, f in vars(d).items() if inspect.isfunction(f) and "return ops." in inspect.getsource(f)}
    assert {getattr(d, n).__name__ for n in wrappers} == set(CALLS)


@pytest.mark.parametrize("name", CALLS)
def test_script(name):
    op, _ = CALLS[name]
    assert "DrissTorch::" + op in str(torch.jit.script(getattr(d, name)).inlined_graph)


@pytest.mark.parametrize("name", CALLS)
def test_symbolic_trace(name):
    op, args = CALLS[name]
    concrete = {p: a for p, a in zip(inspect.signature(getattr(d, name)).parameters, args) if not isinstance(a, torch.Tensor)}
    concrete.update((p.name, p.default) for p in inspect.signature(getattr(d, name)).parameters.values() if p.default is not p.empty)
    graph = torch.fx.symbolic_trace(getattr(d, name), concrete_args=concrete).graph
    assert getattr(torch.ops.DrissTorch, op) in [n.target for n in graph.nodes if n.op == "call_function"]


@pytest.mark.parametrize("name", CALLS)
def test_function_mode(name):
    op, args = CALLS[name]
    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return args[0]

    with Watch():
        getattr(d, name)(*args)
    assert getattr(torch.ops.DrissTorch, op) in seen
