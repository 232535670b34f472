"""autograd Functions of the deformable convolution, mirroring the reference's
`ConvOffset3dFunction` (deform3d/deform_conv3d_functions/deform_conv3d_function.py:7-77) and
`ConvOffset2dFunction` (deform2d_double/deform_conv2d_functions/deform_conv2d_function.py:7-77;
deform2d/deform_conv2d_functions/deform_conv2d_function.py:7-57 is its float, dilation-1,
group-1, bias-free subset).

Same call shape: `Fn.apply(inputs, offset, weight, bias=None, stride, padding, dilation,
channel_per_group=1, group=1)` (plus two optional trailing arguments: `standard_output_size`, see
`output_size`, and `oob_offset_grad`: 'reference' keeps the 3-D kernels' +-|grad column| term in
grad_offset for samples outside the input (deform3d/lib/deform_conv3d_cuda_kernel.cu:470-481), 'zero'
leaves it out, which makes grad_offset the derivative of the forward pass everywhere); same
dilation-blind output size by default; same shape checks and messages
as the reference's `shape_check` (deform3d/lib/deform_conv3d_cuda.cpp:24-87), raised as
RuntimeError.  Differences: no column workspace is kept (the kernels never build one),
float32 and float64 are served by the same class for both 2-D and 3-D, and gradients that are
not required come back as None instead of crashing (the reference wraps None in Variable, :76).
All tensors must live on one MI355X; there is no CPU path.

`apply` hands over to the C++ extension (csrc/dcn_torch.cpp), which checks the call, runs the
operators and records the backward node.  A call under `torch.jit.trace` and a class derived from one of
the Functions go through PyTorch's own `Function.apply` and the class's `forward` and `backward`, which run
the same operators; so do arguments with forward-mode tangents and calls under functorch transforms, which
`Function.apply` refuses (the layers have no forward-mode derivative).
"""
import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable

from . import _lib


def output_size(in_sizes, kernel, stride, padding, dilation=None, standard=False):
    """The reference formula, dilation not included (deform3d/lib/deform_conv3d_cuda.cpp:15-17;
    deform_conv3d_function.py:26-27).  `standard=True` gives the usual dilation-aware size
    `(in + 2p - d(k-1) - 1) // s + 1` instead (the one the reference's plain convolution uses,
    conv2d/lib/conv2d_cuda.cpp:20-22): with it every tap of every output position starts inside
    the padded input, as in an ordinary convolution."""
    if standard:
        dilation = dilation if dilation is not None else (1,) * len(kernel)
        return tuple((i + 2 * p - d * (k - 1) - 1) // s + 1
                     for i, k, s, p, d in zip(in_sizes, kernel, stride, padding, dilation))
    return tuple((i + 2 * p - k) // s + 1 for i, k, s, p in zip(in_sizes, kernel, stride, padding))


def shape_check(nd, inputs, weight, offset, output_shape, channel_per_group, group, stride, padding,
                dilation=None, standard=False):
    """The reference's shape_check with its messages: the checks that every call of a layer goes through."""
    _lib.native().shape_check(nd, inputs, weight, offset, output_shape, stride, padding, 1 if dilation is None else dilation,
                              channel_per_group, group, standard)


# Arguments and workspace of a C-ABI call, for callers of libdcn_amd.so itself.
def _geom(nd, inputs, weight, out_sizes, stride, padding, dilation, channel_per_group, group):
    return ([inputs.size(0), inputs.size(1), weight.size(0)] + list(inputs.shape[2:]) + list(out_sizes) +
            list(weight.shape[2:]) + list(padding) + list(stride) + list(dilation) + [channel_per_group, group])


def _workspace_bytes(inputs, weight, group, out_sizes, channel_per_group):
    L = _lib.load()
    kV = inV = outV = 1
    for k in weight.shape[2:]:
        kV *= k
    for v in inputs.shape[2:]:
        inV *= v
    for v in out_sizes:
        outV *= v
    return int(L.dcn_workspace_bytes_for(inputs.element_size(), inputs.size(0), inputs.size(1), weight.size(0), inV, outV,
                                         kV, group, channel_per_group))


def _workspace(inputs, weight, group, out_sizes, channel_per_group):
    nbytes = _workspace_bytes(inputs, weight, group, out_sizes, channel_per_group)
    return torch.empty(max(nbytes, 1), dtype=torch.uint8, device=inputs.device), nbytes


def _oob_zero(oob_offset_grad):
    if oob_offset_grad not in ("reference", "zero"):
        raise ValueError("oob_offset_grad must be 'reference' or 'zero'")
    return oob_offset_grad == "zero"


class _ConvOffsetNdFunction(Function):
    ND = 0

    @classmethod
    def _fwd(cls, ctx, inputs, offset, weight, bias, *layer):
        ctx.layer = layer[:-1] + (_oob_zero(layer[-1]),)
        ctx.has_bias = bias is not None
        ctx.save_for_backward(inputs, offset, weight)
        return _lib.native().conv_offset_forward(cls.ND, inputs, offset, weight, bias, *ctx.layer)

    @classmethod
    def _bwd(cls, ctx, grad_output):
        inputs, offset, weight = ctx.saved_tensors
        need = ctx.needs_input_grad
        # grad_input and grad_offset come out of one kernel, as in the reference (:52)
        gi, go, gw, gb = _lib.native().conv_offset_backward(cls.ND, inputs, offset, weight, grad_output, *ctx.layer, need[0] or need[1],
                                                            need[2], ctx.has_bias and need[3])
        return (gi if need[0] else None, go if need[1] else None, gw, gb) + (None,) * 7


class ConvOffset3dFunction(_ConvOffsetNdFunction):
    ND = 3

    @classmethod
    def apply(cls, inputs, offset, weight, bias=None, stride=(1, 1, 1), padding=(0, 0, 0), dilation=(1, 1, 1),
              channel_per_group=1, group=1, standard_output_size=False, oob_offset_grad="reference"):
        if cls is ConvOffset3dFunction:
            out = _lib.native().conv_offset(3, inputs, offset, weight, bias, stride, padding, dilation, channel_per_group, group,
                                            standard_output_size, _oob_zero(oob_offset_grad))
            if out is not NotImplemented:
                return out
        return super().apply(inputs, offset, weight, bias, stride, padding, dilation, channel_per_group, group,
                             standard_output_size, oob_offset_grad)

    @staticmethod
    def forward(ctx, inputs, offset, weight, bias=None, stride=(1, 1, 1), padding=(0, 0, 0), dilation=(1, 1, 1),
                channel_per_group=1, group=1, standard_output_size=False, oob_offset_grad="reference"):
        return ConvOffset3dFunction._fwd(ctx, inputs, offset, weight, bias, stride, padding, dilation,
                                         channel_per_group, group, standard_output_size, oob_offset_grad)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_output):
        return ConvOffset3dFunction._bwd(ctx, grad_output)


class ConvOffset2dFunction(_ConvOffsetNdFunction):
    ND = 2

    @classmethod
    def apply(cls, inputs, offset, weight, bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1),
              channel_per_group=1, group=1, standard_output_size=False, oob_offset_grad="reference"):
        if cls is ConvOffset2dFunction:
            out = _lib.native().conv_offset(2, inputs, offset, weight, bias, stride, padding, dilation, channel_per_group, group,
                                            standard_output_size, _oob_zero(oob_offset_grad))
            if out is not NotImplemented:
                return out
        return super().apply(inputs, offset, weight, bias, stride, padding, dilation, channel_per_group, group,
                             standard_output_size, oob_offset_grad)

    @staticmethod
    def forward(ctx, inputs, offset, weight, bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1),
                channel_per_group=1, group=1, standard_output_size=False, oob_offset_grad="reference"):
        return ConvOffset2dFunction._fwd(ctx, inputs, offset, weight, bias, stride, padding, dilation,
                                         channel_per_group, group, standard_output_size, oob_offset_grad)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_output):
        return ConvOffset2dFunction._bwd(ctx, grad_output)
