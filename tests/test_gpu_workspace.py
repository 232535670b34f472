"""Workspaces smaller than the queried one, down to the least that the operators have always taken: the kernels that need less of it,
against the oracle, without a write past the end."""
import ctypes

import pytest
import torch

from deform_conv3d_pytorch_op_amd import _lib
from deform_conv3d_pytorch_op_amd.functions import _geom, _workspace_bytes
from oracle import dcn_oracle as orc
from tests.cases import make_case

pytestmark = pytest.mark.gpu

SUFFIX = {torch.float32: "f32", torch.bfloat16: "bf16"}
ONCE = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -9}       # a result rounded to the storage format


def _up(v, to):
    return (v + to - 1) // to * to


def _least_data_bytes(c):
    """Packed weights of the kernels on the float32 instructions and two channels-last float32 tensors."""
    w, G, cpg = c["w"], c["groups"], c["cpg"]
    M, Cg, kV = w.shape[0] // G, w.shape[1], w[0, 0].numel()
    steps = (M + 1) // 2
    mk = next((k for k in (8, 16, 32, 64) if k >= steps), 0)
    plain = (G * kV + 8) * max(_up(steps, 8) * 2 + 2, mk * 2) * (Cg + 32)
    packed = max((G * Cg // n + G * Cg // cpg + G + 1) * (-(-kV // (32 // n))) * _up(steps, 16) * 64 for n in (4, 8, 16))
    return _up(max(plain, packed) * 4, 256) + 2 * _up(c["x"].numel() * 4, 256)


def _call(fn, c, tensors, ws_bytes):
    """fn on a workspace of ws_bytes, all of it and what lies behind it filled with NaN first."""
    geom = _geom(c["nd"], c["x"], c["w"], c["outs"], c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    ws = torch.full((ws_bytes // 4 + 1024,), float("nan"), device="cuda")
    rc = fn(*(t.data_ptr() for t in tensors), *geom, ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.isnan(ws[ws_bytes // 4:]).all()
    return rc


def _oracle(c):
    """In float32 with double sums: the coordinates are then those of the kernels."""
    d = {k: c[k].float() for k in ("x", "off", "w", "gout")}
    return [t.double() for t in orc.backward(d["x"], d["off"], d["w"], d["gout"], None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])[:3]]


# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): chunks of 16, 8 and 4 channels, more output channels than operand
# registers, several groups, blocks of 128 positions, a single tap
DATA = [(2, 2, 33, 70, (17, 19), 3, 1, 1, 1, 33, 1, 1.5), (2, 1, 12, 24, (18, 18), 3, 2, 1, 1, 4, 2, 2.0), (3, 1, 24, 40, (6, 9, 17), 3, 1, 1, 1, 24, 1, 1.5),
        (3, 1, 16, 130, (6, 15, 17), 3, (1, 2, 2), 1, 1, 8, 1, 2.0), (3, 2, 18, 20, (5, 9, 11), 1, 1, 0, 1, 9, 1, 1.0)]


@pytest.mark.parametrize("dtype", list(SUFFIX), ids=SUFFIX.values())
@pytest.mark.parametrize("spec", DATA, ids=lambda s: "%dd-%d-%d-k%d" % (s[0], s[2], s[3], s[5]))
def test_backward_input_offset(spec, dtype):
    """2-norm: grad_input rounded to 32-bit fixed point (1e-4 of its largest values at most), grad_offset a chain of float32 sums."""
    print("data", spec, dtype, flush=True)
    L, c = _lib.load(), make_case(*spec, dtype=dtype, seed=51, bias=False)
    fn = getattr(L, "dcn%dd_backward_input_offset_%s" % (c["nd"], SUFFIX[dtype]))
    x, w, off, gout = (c[k].cuda() for k in ("x", "w", "off", "gout"))
    copies = 0 if dtype == torch.float32 else sum(_up(t.numel() * 4, 256) for t in (x, w, off, gout, x, off))
    least, full = copies + _least_data_bytes(c), _workspace_bytes(x, w, c["groups"], c["outs"], c["cpg"])
    assert least < full
    got = {}
    for ws_bytes in (least, least + 1024, full):
        gin, goff = torch.zeros_like(x), torch.full_like(off, float("nan"))
        assert _call(fn, c, (x, w, off, gout, gin, goff), ws_bytes) == 0, L.dcn_last_error()
        got[ws_bytes] = gin, goff
        for g, want, tol in zip((gin, goff), _oracle(c), (1e-4, 1e-5)):
            err = ((g.cpu().double() - want).norm() / want.norm()).item()
            print("  %d of %d bytes: relative 2-norm error %.2e" % (ws_bytes, full, err), flush=True)
            assert err <= tol + ONCE[dtype]
    if dtype == torch.float32 and spec[5] > 1:      # two kernels, whose sums are rounded differently
        assert not torch.equal(got[least][1], got[full][1])
    gin, goff = torch.full_like(x, 7.0), torch.full_like(off, 7.0)
    assert _call(fn, c, (x, w, off, gout, gin, goff), least - 256) == -2
    assert (goff == 7.0).all()


# few channels and many positions, so that the channels-last copy of grad_output and the partial tiles leave no room for it in operand order
WEIGHT = [(3, 2, 4, 66, (13, 32, 33), 3, 1, 1, 1, 4, 1, 1.5), (3, 3, 4, 40, (11, 33, 31), 3, 1, 1, 1, 2, 1, 1.0)]


@pytest.mark.parametrize("spec", WEIGHT, ids=lambda s: "%dd-%d-%d" % (s[0], s[2], s[3]))
def test_backward_weight(spec):
    """2-norm: chains of float32 sums over up to a few hundred steps, each off by half a unit in the last place: below
    2^-24 * 64 = 4e-6."""
    print("weight", spec, flush=True)
    L, c = _lib.load(), make_case(*spec, dtype=torch.float32, seed=52, bias=False)
    x, w, off, gout = (c[k].cuda() for k in ("x", "w", "off", "gout"))
    full = _workspace_bytes(x, w, c["groups"], c["outs"], c["cpg"])
    kV, positions = w[0, 0].numel(), gout[:, 0].numel()
    partials = -(-2560 // kV) * w.numel() * 4                               # one channel tile, one chunk of output channels
    copies = _up(x.numel() * 4, 256) + _up(gout.numel() * 4, 256)
    least = copies + _up(partials, 256)
    assert least < _up(x.numel() * 4, 256) + positions * w.shape[0] * 6      # (three bfloat16 parts of grad_output)
    got = {}
    for ws_bytes in (least, full):
        gw = torch.zeros_like(w)
        assert _call(L.dcn3d_backward_weight_f32, c, (x, off, gout, gw), ws_bytes) == 0, L.dcn_last_error()
        got[ws_bytes] = gw
        want = _oracle(c)[2]
        err = ((gw.cpu().double() - want).norm() / want.norm()).item()
        print("  %d of %d bytes: relative 2-norm error %.2e" % (ws_bytes, full, err), flush=True)
        assert err <= 4e-6
    assert not torch.equal(got[least], got[full])                           # two kernels
    assert _call(L.dcn3d_backward_weight_f32, c, (x, off, gout, torch.zeros_like(w)), copies) == -2


# served by the 16-bit kernels; grad_weight on float copies (odd channels); the other gradients (a halo past every block); all of them; a
# single tap of more output channels than operand registers
LAYERS = [(3, 1, 24, 40, (6, 9, 17), 3, 1, 1, 1, 24, 1, 1.5), (2, 2, 33, 70, (17, 19), 3, 1, 1, 1, 33, 1, 1.5), (3, 1, 8, 16, (9, 9, 9), 5, 1, 4, 2, 8, 1, 1.0),
          (3, 2, 7, 12, (9, 9, 9), 5, 1, 4, 2, 7, 1, 1.0), (2, 1, 16, 300, (18, 19), 1, 1, 0, 1, 16, 1, 1.0)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64], ids=["bf16", "f16", "f32", "f64"])
@pytest.mark.parametrize("spec", LAYERS, ids=lambda s: "%dd-%d-%d-k%d" % (s[0], s[2], s[3], s[5]))
def test_layer_backward(spec, dtype):
    """The one-call backward pass on exactly the queried bytes."""
    print("layer", spec, dtype, flush=True)
    L, c = _lib.load(), make_case(*spec, dtype=dtype, seed=53, bias=False)
    x, w, off, gout = (c[k].cuda() for k in ("x", "w", "off", "gout"))
    nd, elem = c["nd"], x.element_size()
    volume = lambda t: t[0, 0].numel()
    query = L.dcn_layer_backward_workspace_bytes
    query.restype, query.argtypes = ctypes.c_size_t, [ctypes.c_int] * 5 + [ctypes.c_size_t] * 2 + [ctypes.c_int] * 3
    ws_bytes = query(elem, nd, x.shape[0], x.shape[1], w.shape[0], volume(x), volume(gout), volume(w), c["groups"], c["cpg"])
    geom = _geom(nd, x, w, c["outs"], c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    ws = torch.full((ws_bytes // 4 + 1024,), float("nan"), device="cuda")
    grads = [torch.full_like(t, 7.0) for t in (x, off, w, w[:, 0, 0, 0].flatten() if nd == 2 else w[:, 0, 0, 0, 0])]
    pointer = lambda t: ctypes.c_void_p(t.data_ptr())
    dt = {torch.float32: 0, torch.float64: 1, torch.bfloat16: 2, torch.float16: 3}[dtype]

    def call(size):
        return L.dcn_layer_backward(nd, dt, *(pointer(t) for t in (x, w, off, gout)), *(pointer(t) for t in grads), (ctypes.c_int * len(geom))(*geom), pointer(ws),
                                    ctypes.c_size_t(size), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.c_uint(0))

    assert call(ws_bytes) == 0, L.dcn_last_error()
    torch.cuda.synchronize()
    assert torch.isnan(ws[ws_bytes // 4:]).all()
    wide = {k: c[k].to(torch.float64 if dtype == torch.float64 else torch.float32) for k in ("x", "off", "w", "gout")}
    want = orc.backward(wide["x"], wide["off"], wide["w"], wide["gout"], None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])[:3]
    want = [t.double() for t in want] + [c["gout"].double().sum(dim=[0] + list(range(2, 2 + nd)))]
    once = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 0.0, torch.float64: 0.0}[dtype]
    tols = [1e-10] * 4 if dtype == torch.float64 else [1e-4 + once, 1e-5 + once, 4e-6 + 2 * once, 4e-6 + once]
    for name, got, ref, tol in zip(("grad_input", "grad_offset", "grad_weight", "grad_bias"), grads, want, tols):
        err = ((got.cpu().double() - ref).norm() / ref.norm()).item()
        print("  %s: relative 2-norm error %.2e" % (name, err), flush=True)
        assert err <= tol
    assert call(1024) == -2
