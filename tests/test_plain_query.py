"""When a step's query may go to a HIP operator through the C ABI: only where nothing but
its values is asked for. A C call is invisible to autograd, to batching and forward-mode
transforms, to a trace and to a mode, so each of them keeps the library's operators."""
from __future__ import annotations

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from winnow_amd import packed_backend as pb


@pytest.fixture
def seen():
    return []


@pytest.fixture
def step(seen):
    def f(x):
        seen.append(pb._plain(x))
        return 2 * x
    return f


class _Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_values_alone(seen, step):
    x = torch.randn(2, 3, dtype=torch.bfloat16)
    step(x)
    with torch.device("cpu"):
        step(x)
    with torch.autocast("cpu", dtype=torch.bfloat16):
        step(x)
    with torch.no_grad():
        step(x.clone().requires_grad_())
    with torch.inference_mode():
        step(x)
    assert seen == [True] * 5


@pytest.mark.parametrize("trace", [
    lambda f, x: torch.jit.trace(f, x, check_trace=False),
    lambda f, x: make_fx(f)(x),
    lambda f, x: make_fx(f, tracing_mode="symbolic")(x),
    lambda f, x: make_fx(f, pre_dispatch=True)(x),
    lambda f, x: torch.vmap(f)(x),
    lambda f, x: torch.func.jvp(f, (x,), (x,)),
    lambda f, x: torch.func.grad(lambda y: f(y).sum())(x),
    lambda f, x: torch.func.functionalize(f)(x),
    lambda f, x: f(x.clone().requires_grad_()),
], ids=["jit", "make_fx", "symbolic", "pre_dispatch", "vmap", "jvp", "grad", "functionalize", "requires_grad"])
def test_traces_and_transforms(seen, step, trace):
    trace(step, torch.randn(2, 3))
    assert seen and not any(seen)


@pytest.mark.parametrize("mode", [_Functions, _Dispatch, lambda: torch.autocast("cpu", dtype=torch.float16)],
                         ids=["function", "dispatch", "autocast"])
def test_modes(seen, step, mode):
    with mode():
        step(torch.randn(2, 3, dtype=torch.bfloat16))
    assert seen == [False]
