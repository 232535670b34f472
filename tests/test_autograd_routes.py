"""Which way a call of the package's Functions goes: the C++ autograd node, or PyTorch's own
`Function.apply` where something other than backward has to know about the call.  On the CPU, with
derived classes whose forward needs no GPU."""
import pytest
import torch


def _functions():
    import deform_conv3d_pytorch_op_amd as dcn
    return [dcn.ConvOffset2dFunction, dcn.ConvOffset3dFunction, dcn.Conv2dFunction]


def _derived(fn):
    class Derived(fn):
        @staticmethod
        def forward(ctx, inputs, *rest):
            ctx.n = 1 + len(rest)
            return inputs * 2

        @staticmethod
        def backward(ctx, grad_output):
            return (grad_output * 2,) + (None,) * (ctx.n - 1)

    return Derived


@pytest.mark.parametrize("fn", _functions(), ids=lambda f: f.__name__)
def test_derived_classes_run_their_own_forward_and_backward(fn):
    x = torch.arange(4.0, requires_grad=True)
    y = _derived(fn).apply(x, torch.zeros(1), torch.zeros(1))
    assert torch.equal(y.detach(), 2 * x.detach())
    y.sum().backward()
    assert torch.equal(x.grad, torch.full((4,), 2.0))


def test_a_trace_being_recorded_goes_through_function_apply():
    """... which the tracer records; it sees nothing of the operators themselves."""
    from deform_conv3d_pytorch_op_amd import _lib
    native, seen = _lib.native(), []

    def f(x):
        seen.append(native.wants_function(x))
        return x + 1
    f(torch.zeros(2))
    torch.jit.trace(f, torch.zeros(2), check_trace=False)
    f(torch.zeros(2))
    assert seen == [False, True, False]


@pytest.mark.parametrize("fn", _functions(), ids=lambda f: f.__name__)
def test_a_traced_call_is_recorded_as_the_function(fn, monkeypatch):
    """On the CPU the call itself is refused (there is no CPU path), by the Function's own forward."""
    import deform_conv3d_pytorch_op_amd as dcn
    nd = 3 if fn is dcn.ConvOffset3dFunction else 2
    x, w = torch.zeros((1, 2) + (4,) * nd), torch.zeros((2, 2) + (1,) * nd)
    args = (x, w) if fn is dcn.Conv2dFunction else (x, torch.zeros((1, 2 * nd) + (4,) * nd), w)
    calls, forward = [], fn.forward
    monkeypatch.setattr(fn, "forward", staticmethod(lambda *a: calls.append(len(a)) or forward(*a)))
    with pytest.raises(RuntimeError, match="GPU"):
        fn.apply(*args)
    assert calls == []
    with pytest.raises(RuntimeError, match="GPU"):
        torch.jit.trace(lambda *t: fn.apply(*t), args, check_trace=False)
    assert len(calls) == 1


@pytest.mark.parametrize("fn", _functions(), ids=lambda f: f.__name__)
@pytest.mark.parametrize("at", range(4))
def test_forward_mode_tangents_are_refused(fn, at, monkeypatch):
    """A tangent on any argument: refused by Function.apply, not dropped."""
    import torch.autograd.forward_ad as fwad
    monkeypatch.setattr(fn, "forward", staticmethod(lambda ctx, inputs, *rest: inputs * 2))       # (needs no GPU)
    args = [torch.ones(3) for _ in range(3 if fn.__name__ == "Conv2dFunction" else 4)]
    at = min(at, len(args) - 1)
    with fwad.dual_level():
        args[at] = fwad.make_dual(args[at], torch.ones(3))
        with pytest.raises(NotImplementedError, match="jvp"):
            fn.apply(*args)


@pytest.mark.parametrize("fn", _functions(), ids=lambda f: f.__name__)
def test_functorch_transforms_are_refused_by_name(fn):
    args = [torch.ones(3) for _ in range(2 if fn.__name__ == "Conv2dFunction" else 3)]
    for call in (lambda: torch.vmap(lambda t: fn.apply(t, *args[1:]))(torch.ones(2, 3)),
                 lambda: torch.func.grad(lambda t: fn.apply(t, *args[1:]).sum())(args[0])):
        with pytest.raises(RuntimeError, match="functorch transforms"):
            call()
