"""The reference's plain convolution package: `Conv2dFunction`
(conv2d/conv2d_functions/conv2d_function.py:7-67) and `Conv2d`
(conv2d/conv2d_modules/conv2d_model.py:11-46).  The float32 forward pass, and the backward pass to the
input at stride 1, have a kernel of their own; the rest, and layers that it is not faster on, run on the
kernels of the 2-D deformable layer with every offset zero (C ABI: conv2d_forward / conv2d_backward_input /
conv2d_backward_weight in include/dcn_amd.h, in place of conv2d/lib/conv2d_cuda.h:17-39).

Same call shape, `Conv2dFunction.apply(inputs, weight, bias=None, stride=(1, 1), padding=(0, 0),
dilation=(1, 1), group=1)`, and the reference's dilation-aware output size
(conv2d_function.py:16-19); backward returns (grad_input, grad_weight, grad_bias, None x 4), with
None for gradients that are not needed (the reference wraps None in Variable there).  float32 and
float64 on one MI355X; there is no CPU path.
"""
import torch
import torch.nn as nn
from torch.autograd import Function
from torch.autograd.function import once_differentiable
from torch.nn.modules.utils import _pair

from . import _lib


class Conv2dFunction(Function):
    @classmethod
    def apply(cls, inputs, weight, bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1), group=1):
        if cls is Conv2dFunction:       # (otherwise through PyTorch's own apply, see functions.py)
            out = _lib.native().conv2d(inputs, weight, bias, stride, padding, dilation, group)
            if out is not NotImplemented:
                return out
        return super().apply(inputs, weight, bias, stride, padding, dilation, group)

    @staticmethod
    def forward(ctx, inputs, weight, bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1), group=1):
        ctx.layer = (stride, padding, dilation, group)
        ctx.has_bias = bias is not None
        ctx.save_for_backward(inputs, weight)
        return _lib.native().conv2d_forward(inputs, weight, bias, *ctx.layer)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_output):
        inputs, weight = ctx.saved_tensors
        need = ctx.needs_input_grad
        gi, gw, gb = _lib.native().conv2d_backward(inputs, weight, grad_output, *ctx.layer, need[0], need[1], ctx.has_bias and need[2])
        return gi, gw, gb, None, None, None, None


class Conv2d(nn.Module):
    """`Conv2d(in_channels, out_channels, kernel_size, stride=1, padding=0, dilation=1, bias=True,
    groups=1)` with parameters `weight` (Kaiming-normal, fan_out) and `bias` (U(-0.1, 0.1)), as
    conv2d/conv2d_modules/conv2d_model.py:11-46; `device` and `dtype` are extra keyword arguments."""

    def __init__(self, in_channels, out_channels, kernel_size, stride=1, padding=0, dilation=1, bias=True, groups=1,
                 device=None, dtype=None):
        super().__init__()
        self.in_channels = in_channels
        self.out_channels = out_channels
        self.kernel_size = _pair(kernel_size)
        self.stride = _pair(stride)
        self.padding = _pair(padding)
        self.dilation = _pair(dilation)
        self.group = groups
        if in_channels % groups != 0:
            raise ValueError('in_channels must be divisible by groups')
        if out_channels % groups != 0:
            raise ValueError('out_channels must be divisible by groups')
        kw = dict(device=device, dtype=dtype)
        self.weight = nn.Parameter(torch.empty(out_channels, in_channels // groups, *self.kernel_size, **kw))
        nn.init.kaiming_normal_(self.weight, mode='fan_out')
        if bias:
            self.bias = nn.Parameter(torch.empty(out_channels, **kw))
            nn.init.uniform_(self.bias, -0.1, 0.1)
        else:
            self.register_parameter('bias', None)

    def forward(self, inputs):
        return Conv2dFunction.apply(inputs, self.weight, self.bias, self.stride, self.padding, self.dilation, self.group)
