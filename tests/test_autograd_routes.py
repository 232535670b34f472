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
