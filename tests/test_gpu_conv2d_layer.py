"""The plain convolution's one-call backward pass at the edges of its dispatch, against torch's convolution in
float64: grad_input as a convolution (stride 1, padding up to dilation * (k - 1)), by the scattering kernel (a
stride, more padding), and layers whose halo no workgroup can hold."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# N, C_in, C_out, in, k, stride, pad, dil, groups
SPECS = [(1, 3, 2, (3, 3), 3, 1, 0, 1, 1), (2, 32, 33, (9, 21), 3, 1, 2, 1, 1), (1, 65, 31, (16, 16), 3, 1, 1, 1, 1),
         (1, 12, 8, (11, 13), (3, 2), 1, (1, 0), (2, 3), 4), (1, 8, 8, (10, 9), 3, 1, 3, 1, 1),
         (2, 16, 24, (15, 18), 3, 2, 1, 1, 2), (1, 130, 96, (20, 33), 5, 1, 2, 1, 1), (1, 40, 72, (7, 40), 1, 1, 0, 1, 2),
         (1, 24, 16, (200, 210), 9, 1, 90, 23, 1)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("spec", SPECS, ids=lambda s: "-".join(str(v) for v in s).replace(" ", ""))
def test_gradients(spec, dtype):
    import deform_conv3d_pytorch_op_amd as dcn
    N, cin, cout, ins, k, stride, pad, dil, groups = spec
    print("conv2d layer", spec, dtype, flush=True)
    torch.manual_seed(3)
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    m = dcn.Conv2d(cin, cout, k, stride, pad, dil, bias=True, groups=groups, device="cuda", dtype=dtype)
    x = torch.randn((N, cin) + ins, dtype=dtype).cuda().requires_grad_()
    y = m(x)
    g = torch.randn(y.shape, dtype=dtype)
    y.backward(g.cuda())
    x64, w64, b64 = (t.detach().cpu().double().requires_grad_() for t in (x, m.weight, m.bias))
    want = F.conv2d(x64, w64, b64, stride, pad, dil, groups)
    want.backward(g.double())
    for name, got, ref in (("y", y, want), ("x", x.grad, x64.grad), ("w", m.weight.grad, w64.grad), ("b", m.bias.grad, b64.grad)):
        err = (got.detach().cpu().double() - ref.detach()).norm() / ref.detach().norm()
        assert err.item() <= tol, (name, err.item())
