"""The operators' direct path (ops._op) on the CPU: an operator whose body reads
its arguments' memory, as the kernels do, gives what the registered custom op
gives for every kind of argument and under everything that interposes on
operators."""

import ctypes
from typing import List, Optional

import numpy as np
import pytest
import torch
from torch.autograd import forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

from fbpinns_amd import ops


def _memory(t):
    """The float32 values at t's data pointer (contiguous tensors with memory
    only, as the operators' own check)."""
    if not t.is_contiguous() or not t.data_ptr():
        raise ops.FbpxError("not contiguous, or no memory")
    return np.frombuffer((ctypes.c_float * t.numel()).from_address(t.data_ptr()), dtype=np.float32)


@ops._op("fbpx_test::axpy", mutates_args=("out",))
def axpy(x: torch.Tensor, ys: List[torch.Tensor], n: List[int], k: int, a: float, flip: bool, out: torch.Tensor,
         scale: Optional[torch.Tensor] = None) -> None:
    v = a * _memory(x) + sum(_memory(y) for y in ys) + k + sum(n)
    if scale is not None:
        v = v * _memory(scale)[0]
    out.detach().numpy()[...] = -v if flip else v


@axpy.custom_op.register_fake
def _(x, ys, n, k, a, flip, out, scale=None):
    return None


def _args(x=None, y=None, scale=None):
    x = torch.tensor([1.0, 2.0, 3.0]) if x is None else x
    y = torch.tensor([0.5, 0.25, 0.125]) if y is None else y
    return [x, [y, y], [1, 2], 3, 2.0, False, torch.zeros(3), scale]


def _both(args):
    a, b = list(args), list(args)
    a[6], b[6] = torch.zeros(3), torch.zeros(3)
    axpy(*a)
    axpy.custom_op(*b)
    return a[6], b[6]


def _negative():
    v = torch._neg_view(torch.tensor([1.0, 2.0, 3.0]))
    assert v.is_neg() and v.is_contiguous()
    return v


def test_plain_call_equals_custom_op():
    got, want = _both(_args())
    assert torch.equal(got, want) and want.abs().sum() > 0
    got, want = _both(_args(scale=torch.tensor([3.0])))
    assert torch.equal(got, want)


@pytest.mark.parametrize("where", ["x", "list", "scale"])
def test_negative_bit(where):
    neg = _negative()
    args = {"x": _args(x=neg), "list": _args(y=neg), "scale": _args(scale=neg)}[where]
    got, want = _both(args)
    assert torch.equal(got, want)


def test_negative_bit_from_autograd():
    """The gradient of a conjugated imaginary part reaches a backward with the
    bit set; the operator called on it reads the gradient's value."""
    seen = []

    class Scale(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x * 2

        @staticmethod
        def backward(ctx, g):
            g = g.contiguous()
            seen.append(g.is_neg())
            out = torch.zeros(())
            axpy(g, [], [], 0, 2.0, False, out)
            return out
    x = torch.tensor(3.0, requires_grad=True)
    loss = Scale.apply(x)
    torch.complex(torch.zeros(()), loss).conj().abs().backward()
    assert seen == [True]
    assert x.grad.item() == 2.0


@pytest.mark.parametrize("where", ["x", "list"])
def test_zero_tensor(where):
    """A zero tensor has no memory, and the custom op gets one expanded element
    for it: refused in both."""
    z = torch._efficientzerotensor(3)
    assert z.is_contiguous() and z.data_ptr() == 0
    for call in (axpy, axpy.custom_op):
        with pytest.raises(ops.FbpxError):
            call(*(_args(x=z) if where == "x" else _args(y=z)))


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_profiler_sees_the_operator():
    args = _args()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as p:
        axpy(*args)
    assert any(e.key == "fbpx_test::axpy" for e in p.key_averages())
    with torch.autograd.profiler.profile() as p:
        axpy(*args)
    assert any(e.key == "fbpx_test::axpy" for e in p.key_averages())


def test_modes_functions_and_subclasses_see_the_operator():
    with _Seen() as seen:
        axpy(*_args())
    assert any("fbpx_test.axpy" in s for s in seen.names)

    names = []

    class Functions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))
    with Functions():
        axpy(*_args())
    assert any("axpy" in s for s in names)

    class Sub(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            names.append("sub " + str(func))
            return super().__torch_function__(func, types, args, kwargs or {})
    axpy(*_args(x=torch.ones(3).as_subclass(Sub)))
    assert any(s.startswith("sub") and "axpy" in s for s in names)


def test_functorch_forward_mode_and_tracing_reach_the_dispatcher():
    """Whatever transforms operators is handed the custom op."""
    from torch.fx.experimental.proxy_tensor import make_fx
    with pytest.raises(RuntimeError):          # no batching rule: refused, as for any custom op
        torch.vmap(lambda x: axpy(x, [], [], 0, 1.0, False, torch.zeros(3)) or x)(torch.ones(2, 3))
    with forward_ad.dual_level():
        d = forward_ad.make_dual(torch.ones(3), torch.ones(3))
        kinds = []
        for call in (axpy, axpy.custom_op):
            try:
                call(d, [], [], 0, 1.0, False, torch.zeros(3))
                kinds.append(None)
            except Exception as e:
                kinds.append(type(e))
        assert kinds[0] is kinds[1]

    def f(x, out):
        axpy(x, [], [], 0, 1.0, False, out)
        return out
    g = make_fx(f, tracing_mode="fake")(torch.ones(3), torch.zeros(3))
    assert "axpy" in g.code


def test_arguments_that_require_a_gradient():
    """Refused by the custom op's autograd in the same way, accepted without
    gradients."""
    x = torch.ones(3, requires_grad=True)
    errors = []
    for call in (axpy, axpy.custom_op):
        out = torch.zeros(3)
        try:
            call(*[x, [], [], 0, 1.0, False, out])
            errors.append((None, out.requires_grad, out.detach().tolist()))
        except RuntimeError as e:
            errors.append((type(e), False, []))
    assert errors[0] == errors[1]
    with torch.no_grad():
        got, want = _both(_args(x=x))
    assert torch.equal(got, want)


def test_inference_tensors_outside_inference_mode():
    with torch.inference_mode():
        x = torch.ones(3)
    got, want = _both(_args(x=x))
    assert torch.equal(got, want)


@pytest.mark.parametrize("at,value", [(2, [1, 2.5]), (2, (1, 2)), (2, ["a"]), (3, 1.5), (3, "a"), (3, True), (4, 2),
                                      (4, "a"), (4, np.float64(2.0)), (5, 1), (0, None), (1, [None]), (7, 1.0)])
def test_schema(at, value):
    """Arguments of another type are converted or refused as the custom op does."""
    results = []
    for call in (axpy, axpy.custom_op):
        args = _args()
        args[at] = value
        try:
            call(*args)
            results.append((None, args[6].tolist()))
        except Exception as e:
            results.append((type(e), args[6].tolist()))
    assert results[0] == results[1], results


@pytest.mark.parametrize("n", [0, 3, 6])
def test_missing_arguments(n):
    kinds = []
    for call in (axpy, axpy.custom_op):
        with pytest.raises(Exception) as e:
            call(*_args()[:n])
        kinds.append(e.type)
    assert kinds[0] is kinds[1]


def test_versions():
    args = _args()
    axpy(*args)
    assert args[6]._version == 1


def test_registrations():
    """The operator's own methods are there, and what they register is used."""
    @ops._op("fbpx_test::fill", mutates_args=("out",))
    def fill(out: torch.Tensor) -> None:
        out.fill_(1.0)
    out = torch.zeros(2)
    fill(out)
    assert out.tolist() == [1.0, 1.0]

    @fill.register_kernel("cpu")
    def _(out):
        out.fill_(2.0)
    fill(out)
    assert out.tolist() == [2.0, 2.0]
    with fill.set_kernel_enabled("cpu", False):
        fill(out)
    assert out.tolist() == [1.0, 1.0]


def test_compilation_sees_the_operator():
    graphs = []

    def backend(gm, example_inputs):
        graphs.append(gm.code)
        return gm.forward

    def f(x, out):
        axpy(x, [x], [1], 2, 1.5, False, out)
        return out + 1
    x, out = torch.ones(3), torch.zeros(3)
    got = torch.compile(f, backend=backend, fullgraph=True)(x, out)
    assert len(graphs) == 1 and "axpy" in graphs[0]
    want = torch.zeros(3)
    axpy.custom_op(x, [x], [1], 2, 1.5, False, want)
    assert torch.equal(got, want + 1)
