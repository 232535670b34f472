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


# The kernel of the plain convolution at the edges of its shapes -- one, two, four and eight row tiles, passes of eight to sixty-four channels
# with remainders, one, two and three tap pairs and a lone tap, strides and dilations, groups, positions that fill no block -- whatever the
# layer's size (DCN_PLAIN=2, read once per process).
PLAIN = [(1, 8, 1, (9, 9), 3, 1, 1, 1, 1), (2, 5, 33, (8, 17), 1, 1, 0, 1, 1), (1, 70, 64, (7, 24), 3, 2, 1, 1, 1), (1, 24, 130, (11, 9), (3, 2), 1, (1, 0), (2, 3), 1),
         (1, 136, 260, (10, 12), 2, 1, 1, 1, 1), (2, 18, 36, (13, 8), 5, (1, 2), 2, 1, 2), (1, 64, 96, (30, 31), 3, 1, 8, 7, 1), (1, 200, 40, (16, 16), 3, 1, 1, 1, 1),
         (1, 12, 300, (9, 10), 3, 1, 2, 2, 4), (3, 1, 1, (1, 1), 1, 1, 0, 1, 1), (1, 40, 16, (20, 22), 7, 1, 3, 1, 1), (1, 16, 520, (9, 9), 1, 1, 0, 1, 1)]


def plain_cases():
    import deform_conv3d_pytorch_op_amd as dcn
    for spec in PLAIN:
        test_gradients(spec, torch.float32)
    # values without bfloat16 parts, and values that are not finite: next to them no result but those that they belong to
    torch.manual_seed(5)
    x = torch.randn(3, 20, 18, 19)
    x[0, 3, 4, 5], x[0, 7, 0, 0] = float("inf"), float("nan")
    x[1] *= 1e-36
    w = torch.randn(40, 20, 3, 3)
    m = dcn.Conv2d(20, 40, 3, 1, 1, bias=False, device="cuda", dtype=torch.float32)
    with torch.no_grad():
        m.weight.copy_(w)
        got = m(x.cuda()).cpu().double()
    want = F.conv2d(x.double(), w.double(), None, 1, 1)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    for n in (1, 2):
        assert ((got[n] - want[n]).norm() / want[n].norm()).item() <= 1e-6
    print("plain cases passed", flush=True)


def test_plain_kernel():
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-u", "-c", "from tests.test_gpu_conv2d_layer import plain_cases; plain_cases()"], cwd=root,
                       env=dict(os.environ, DCN_PLAIN="2", DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and "plain cases passed" in r.stdout, r.stdout[-3000:]
    assert r.stdout.count("dcn plain convolution") >= 2 * len(PLAIN) - 4      # (grad_input of layers with a stride or more padding than span is no convolution)
    assert "dcn forward:" not in r.stdout
    for rows in ("1 wavefronts along the rows, 1 row", "2 wavefronts along the rows, 1 row", "4 wavefronts along the rows, 1 row", "4 wavefronts along the rows, 2 row"):
        assert rows in r.stdout


# Layers of long sums that the kernel takes, of each variant; the other kernels share most of their positions among wavefronts or workgroups.  The last one's values are all positive.
LONG = [(1, 47, 256, 69, 86, 3), (8, 19, 256, 14, 63, 3), (2, 45, 128, 40, 89, 3), (2, 21, 64, 67, 75, 5), (16, 440, 64, 50, 25, 3), (16, 23, 15, 78, 66, 3), (8, 374, 37, 33, 89, 1)]


def long_sums():
    import deform_conv3d_pytorch_op_amd as dcn
    for n, (N, cin, cout, h, w, k) in enumerate(LONG):
        torch.manual_seed(n)
        x, wt = torch.randn(N, cin, h, w), torch.randn(cout, cin, k, k)
        if n == len(LONG) - 1:
            x, wt = x.abs(), wt.abs()
        got = dcn.Conv2dFunction.apply(x.cuda(), wt.cuda(), None, 1, k // 2, 1, 1).cpu().double()
        want = F.conv2d(x.double(), wt.double(), None, 1, k // 2)
        print("error %.4e" % ((got - want).norm() / want.norm()).item(), flush=True)


def test_plain_kernel_is_as_exact_as_the_others():
    """2-norm against float64, at most that of the kernels of the deformable layer (DCN_PLAIN=0), whose sums are those of the float32 operator."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    errors = {}
    for knob in ("0", "1"):
        r = subprocess.run([sys.executable, "-u", "-c", "from tests.test_gpu_conv2d_layer import long_sums; long_sums()"], cwd=root,
                           env=dict(os.environ, DCN_PLAIN=knob, DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
        assert r.returncode == 0, r.stdout[-3000:]
        errors[knob] = [float(l.split()[1]) for l in r.stdout.splitlines() if l.startswith("error ")]
        assert len(errors[knob]) == len(LONG) and r.stdout.count("dcn plain convolution") == (len(LONG) if knob == "1" else 0)
    print(errors, flush=True)
    for spec, other, own in zip(LONG, errors["0"], errors["1"]):
        assert own <= other, (spec, own, other)
