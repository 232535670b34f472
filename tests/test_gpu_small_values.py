"""float32 operands so small that their bfloat16 parts lose bits: results as exact as for ordinary ones."""
import pytest
import torch
import torch.nn.functional as F

from tests.cases import make_case
from tests.test_gpu_split import _forward, _oracle

pytestmark = pytest.mark.gpu

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): shared columns, up to four row tiles, 3-D
SPECS = {"2d-split": (2, 1, 20, 65, (19, 33), 3, 1, 1, 1, 20, 1, 1.5), "2d-shared": (2, 2, 40, 257, (40, 33), 3, 1, 1, 1, 20, 1, 1.0),
         "3d-groups": (3, 1, 12, 64, (5, 9, 10), 3, 1, 1, 1, 4, 1, 1.5), "3d-far": (3, 1, 16, 34, (6, 12, 10), 2, 1, 1, 1, 16, 2, 6.0)}


@pytest.mark.parametrize("spec", SPECS.values(), ids=SPECS)
@pytest.mark.parametrize("what,exponent", [("x", 111), ("x", 118), ("x", 124), ("w", 111), ("w", 118), ("w", 126), ("w", 140)])
def test_scaled_operand(spec, what, exponent):
    """One operand times 2^-exponent, the other times a power of two that keeps the results normal numbers (scaling
    both is exact): the error against float64 that ordinary operands have, see test_edges_and_accuracy.
    (x down to 2^-124: below that the samples themselves are subnormal.)"""
    print("small", spec, what, exponent, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=21)
    c["b"] = None
    c[what] = c[what] * 2.0 ** -exponent
    other = "w" if what == "x" else "x"
    c[other] = c[other] * 2.0 ** (10 if exponent < 130 else 30)
    got, want = _forward(c).cpu().double(), _oracle(c)
    assert want.abs().median().item() > 2.0 ** -126
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= 2e-6


def test_one_small_row_and_one_small_region():
    """Small results beside ordinary ones: each output channel and each position on its own."""
    c = make_case(2, 1, 16, 40, (24, 40), 3, 1, 1, 1, 16, 1, 0.9, dtype=torch.float32, seed=22)
    c["b"] = None
    c["w"][7] *= 2.0 ** -116
    c["x"][..., 20:] *= 2.0 ** -118
    print("small row and region", flush=True)
    got, want = _forward(c).cpu().double(), _oracle(c)
    for part in ((slice(None), slice(None), slice(None), slice(24, None)), (slice(None), 7, slice(None), slice(0, 16)), (slice(None), 9)):
        g, w = got[part], want[part]
        assert ((g - w).norm() / w.norm()).item() <= 2e-6


def test_plain_convolution_and_its_grad_input():
    import deform_conv3d_pytorch_op_amd as dcn
    print("small conv2d", flush=True)
    g = torch.Generator().manual_seed(3)
    x, w, go = (torch.randn(s, generator=g) for s in ((2, 24, 17, 19), (40, 24, 3, 3), (2, 40, 17, 19)))
    x, w, go = x * 2.0 ** 8, w * 2.0 ** -119, go * 2.0 ** 8
    xg = x.cuda().requires_grad_()
    y = dcn.Conv2dFunction.apply(xg, w.cuda(), None, 1, 1, 1, 1)
    y.backward(go.cuda())
    xr = x.double().requires_grad_()
    yr = F.conv2d(xr, w.double(), padding=1)
    yr.backward(go.double())
    for got, want in ((y.detach(), yr.detach()), (xg.grad, xr.grad)):
        assert ((got.cpu().double() - want).norm() / want.norm()).item() <= 2e-6
