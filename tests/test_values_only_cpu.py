"""Calls that ask torch for more than values (tangents, transforms, tracing,
modes, subclasses) keep to torch's ops: the condition under which the fused
kernels stand in for them, and the projections under it."""
import pytest
import torch
import torch.autograd.forward_ad as fwad
import torch.nn.functional as F
from torch._subclasses import FakeTensorMode
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from tinyvllm.kernels._extension import values_only
from tinyvllm.layers import PackedLinear, SplitKLinear


def test_plain_calls():
    x = torch.randn(2, 4)
    assert not values_only(x)  # gradients enabled
    with torch.no_grad():
        assert values_only(x, torch.nn.Parameter(x))
        with torch.device("cpu"):  # a default device asks for nothing
            assert values_only(x)
    with torch.inference_mode():
        assert values_only(x)


class _Subclass(torch.Tensor):
    pass


class _Sees(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_calls_for_more_than_values():
    x = torch.randn(2, 4)
    seen = {}

    def note(name, t):
        seen[name] = values_only(t)
        return t * 1

    with torch.no_grad():
        with fwad.dual_level():
            note("dual level", x)
        torch.func.vmap(lambda t: note("vmap", t))(x)
        torch.func.jvp(lambda t: note("jvp", t), (x,), (x,))
        torch.func.functionalize(lambda t: note("functionalize", t))(x)
        torch.jit.trace(lambda t: note("trace", t), (x,), check_trace=False)
        with FlopCounterMode(display=False):
            note("dispatch mode", x)
        with _Sees():
            note("function mode", x)
        note("subclass", x.as_subclass(_Subclass))
        with FakeTensorMode():
            note("fake", torch.empty(2, 4, device="cuda"))
    assert seen and not any(seen.values()), seen


@pytest.mark.parametrize("build", [
    lambda: PackedLinear(64, (64, 64), device="cuda", dtype=torch.bfloat16),
    lambda: SplitKLinear(64, 96, device="cuda", dtype=torch.bfloat16)])
def test_projections_trace_under_fake_tensors(build):
    """Shapes of a GPU model are traced without a GPU."""
    with FakeTensorMode(), torch.no_grad():
        layer = build()
        y = layer(torch.empty(3, 64, device="cuda", dtype=torch.bfloat16))
        y = y.materialize() if hasattr(y, "materialize") else y
        assert y.shape == (3, layer.weight.shape[0]) and y.dtype == torch.bfloat16


def test_projections_under_compile():
    """A compiled program holds the projection itself, without a graph break."""
    layer = PackedLinear(64, (64, 64))
    x = torch.randn(3, 64)
    with torch.no_grad():
        y = torch.compile(lambda t: layer(t) + 1, backend="eager", fullgraph=True)(x)
        torch.testing.assert_close(y, F.linear(x, layer.weight) + 1)
