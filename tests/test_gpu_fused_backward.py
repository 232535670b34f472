"""backward_fused_kernel: edges of its tiles, chunks and block shapes, and the operands that bfloat16 parts do not hold."""
import ast
import os
import re
import subprocess
import sys

import pytest
import torch

from oracle import dcn_oracle as orc
from tests.cases import make_case

pytestmark = pytest.mark.gpu

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): steps of 16 output channels and their remainders;
# chunks of 16, 8 and 4 channels and short ones; two and several tiles to a contraction (9, 25 taps); blocks of 128
# positions (strides in 3-D); wide halos and samples past every halo; a deformable group over two convolution groups.  Single taps
# take backward_input_halo_kernel, but for 16-bit storage of more than 256 output channels (EDGES16).
EDGES = [
    (2, 1, 16, 1, (17, 16), 3, 1, 1, 1, 16, 1, 1.5), (2, 1, 17, 15, (9, 33), 3, 1, 1, 1, 17, 1, 1.5),
    (2, 1, 33, 16, (16, 17), 3, 1, 1, 1, 33, 1, 3.5), (2, 2, 15, 17, (11, 12), 3, 1, 1, 1, 15, 1, 1.0),
    (2, 1, 9, 65, (20, 18), 3, 2, 1, 1, 9, 1, 2.0), (2, 1, 40, 129, (12, 13), 3, 1, 1, 1, 20, 1, 2.0),
    (2, 1, 24, 34, (18, 18), 5, 1, 2, 1, 24, 1, 2.0), (2, 1, 18, 20, (13, 11), 1, 1, 0, 1, 18, 1, 1.5),
    (2, 1, 24, 32, (14, 14), 3, 1, 1, 1, 24, 2, 9.0), (2, 1, 8, 8, (24, 24), 3, 3, 1, 2, 2, 1, 2.0),
    (3, 1, 8, 16, (5, 9, 10), 3, 1, 1, 1, 8, 1, 1.5), (3, 1, 9, 33, (4, 8, 9), 3, 1, 1, 1, 9, 1, 3.5),
    (3, 1, 12, 80, (9, 21, 19), 3, 2, 1, 1, 12, 1, 2.0), (3, 1, 16, 130, (6, 15, 17), 3, (1, 2, 2), 1, 1, 8, 1, 2.0),
    (3, 1, 20, 17, (5, 9, 9), 2, 1, 1, 1, 10, 1, 6.0), (3, 1, 8, 24, (9, 9, 9), 3, 1, 2, 2, 4, 2, 2.5),
    (3, 1, 10, 7, (6, 5, 40), 1, 1, 0, 1, 5, 1, 1.5),
]
EDGES16 = [
    (2, 1, 18, 257, (13, 11), 1, 1, 0, 1, 18, 1, 1.5), (2, 1, 9, 264, (17, 16), 1, 2, 0, 1, 9, 1, 1.5), (2, 2, 12, 300, (9, 33), 1, 1, 0, 1, 3, 1, 3.5),
    (3, 1, 10, 257, (5, 6, 9), 1, 1, 0, 1, 5, 1, 1.5), (3, 1, 13, 272, (4, 9, 20), 1, (1, 2, 2), 0, 1, 13, 1, 6.0), (3, 1, 16, 530, (4, 8, 8), 1, 1, 0, 1, 8, 2, 1.5),
]


def _gradients(c):
    """grad_input, grad_offset"""
    import deform_conv3d_pytorch_op_amd as dcn
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    x, off, w = (c[k].cuda().requires_grad_(k != "w") for k in ("x", "off", "w"))
    fn.apply(x, off, w, None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"]).backward(c["gout"].cuda())
    return x.grad.cpu().double(), off.grad.cpu().double()


def _oracle(c):
    """In float32 with double sums: the coordinates are then those of the kernel."""
    d = {k: c[k].float() for k in ("x", "off", "w", "gout")}
    return [t.double() for t in orc.backward(d["x"], d["off"], d["w"], d["gout"], None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])[:2]]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("spec", EDGES, ids=lambda s: "%dd-%d-%d-k%d-cpg%d" % (s[0], s[2], s[3], s[5], s[9]))
def test_edges(spec, dtype):
    """2-norm: grad_input is rounded to 32-bit fixed point (1e-4 of its largest values at most), grad_offset a chain of
    float32 sums over the channels; 16-bit results are rounded once more (2^-9 and 2^-12 of each value)."""
    print("edges", spec, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=31, bias=False)
    once = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    for got, want, tol in zip(_gradients(c), _oracle(c), (1e-4, 1e-5)):
        err = ((got - want).norm() / want.norm()).item()
        print("  relative 2-norm error %.2e" % err, flush=True)
        assert err <= tol + once


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("spec", EDGES16, ids=lambda s: "%dd-%d-%d-k%d-cpg%d" % (s[0], s[2], s[3], s[5], s[9]))
def test_edges_of_single_taps(spec, dtype):
    test_edges(spec, dtype)


def test_kernels_of_the_edges():
    """backward_fused_kernel runs what these tests are for (the trace of the plans, in a process of its own: the knob is read once)."""
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", __file__, "-q", "-x", "-s", "-m", "gpu", "-k", "test_edges", "--timeout", "120",
                        "--timeout-method", "thread"], cwd=os.path.dirname(here), env=dict(os.environ, DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    cases = r.stdout.split("edges (")[1:]
    assert len(cases) == 3 * len(EDGES) + 2 * len(EDGES16)
    for case in cases:
        spec = ast.literal_eval("(" + case[:case.index(" torch.")])
        launches = re.findall(r"dcn backward_input_offset: launch.*", case)
        print(spec, launches, flush=True)
        one_tap = spec[5] == 1 and spec not in EDGES16
        assert launches and all(("(halo kernel)" in l) == one_tap for l in launches), spec


@pytest.mark.parametrize("spec", [EDGES[5], EDGES[10], EDGES[13]], ids=["2d", "3d", "3d-strided"])
@pytest.mark.parametrize("what,exponent", [("gout", 60), ("gout", 111), ("gout", 118), ("w", 111), ("w", 118), ("w", 126), ("w", 140)])
def test_small_operands(spec, what, exponent):
    """One operand times 2^-exponent, the other times a power of two that keeps the gradients normal numbers: as exact as
    ordinary operands, whose errors test_edges bounds."""
    print("small", spec, what, exponent, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=32, bias=False)
    c[what] = c[what] * 2.0 ** -exponent
    other = "w" if what == "gout" else "gout"
    c[other] = c[other] * 2.0 ** (10 if exponent < 130 else 30)
    for got, want, tol in zip(_gradients(c), _oracle(c), (1e-4, 1e-5)):
        assert want.abs().max().item() > 2.0 ** -122
        err = ((got - want).norm() / want.norm()).item()
        print("  relative 2-norm error %.2e" % err, flush=True)
        assert err <= tol


@pytest.mark.parametrize("spec", [EDGES[5], EDGES[7], EDGES[13], EDGES[16]], ids=["2d", "2d-k1", "3d-strided", "3d-k1"])
@pytest.mark.parametrize("w,gout", [(62, 0), (66, 0), (90, 0), (98, 0), (101, 0), (120, 10), (140, 30), (55, -55), (30, -58), (58, -30), (0, -58)])
def test_small_weights(spec, w, gout):
    """Weights times 2^-w and grad_output times 2^gout, on both sides of the lines between cells and global memory (products of about
    2^-100) and of squares that underflow (weights below 2^-63): gradients that are normal numbers are as exact as ordinary ones."""
    print("small weights", spec, w, gout, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=35, bias=False)
    c["w"] = c["w"] * 2.0 ** -w
    c["gout"] = c["gout"] * 2.0 ** gout
    for got, want, tol in zip(_gradients(c), _oracle(c), (1e-4, 1e-5)):
        assert want.abs().max().item() > 2.0 ** -122
        err = ((got - want).norm() / want.norm()).item()
        print("  relative 2-norm error %.2e" % err, flush=True)
        assert err <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("share", [0.002, 0.3], ids=["few", "many"])
@pytest.mark.parametrize("spec", [(3, 1, 8, 16, (9, 12, 14), 3, 1, 1, 1, 8, 1, 1.0), (3, 2, 15, 20, (9, 17, 15), 3, 1, 1, 1, 5, 1, 1.0),
                                  (3, 1, 17, 40, (10, 21, 19), 3, 2, 1, 1, 17, 1, 1.0), (3, 1, 4, 8, (9, 11, 12), 2, 1, 1, 1, 2, 1, 1.0),
                                  (2, 1, 33, 48, (30, 34), 3, 1, 1, 1, 33, 1, 1.0), (2, 2, 12, 24, (26, 31), 3, 2, 1, 1, 6, 2, 1.0)],
                         ids=lambda s: "%dd-%d-cpg%d" % (s[0], s[2], s[9]))
def test_samples_past_the_halo(spec, share, dtype):
    """Single samples, and most of a tap slot's, that reach past the halo, with full and short chunks of every width: grad_offset of those
    samples by themselves (bounds as in test_edges), and grad_input."""
    print("past the halo", spec, share, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=36, bias=False)
    g = torch.Generator().manual_seed(37)
    far = torch.rand(c["off"].shape, generator=g) < share
    wide = (torch.randint(0, 2, c["off"].shape, generator=g) * 2 - 1) * (7 + 2 * torch.rand(c["off"].shape, generator=g))
    c["off"] = torch.where(far, wide.to(dtype), c["off"])
    nd, taps = spec[0], spec[5] ** spec[0]
    of_sample = far.view(spec[1], -1, taps, nd, *c["outs"]).any(3, keepdim=True).expand(-1, -1, -1, nd, *c["outs"]).reshape(far.shape)
    once = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    (gin, goff), (win, woff) = _gradients(c), _oracle(c)
    assert woff[of_sample].norm() > 0
    for got, want, tol in ((gin, win, 1e-4), (goff[of_sample], woff[of_sample], 1e-5), (goff, woff, 1e-5)):
        err = ((got - want).norm() / want.norm()).item()
        print("  relative 2-norm error %.2e" % err, flush=True)
        assert err <= tol + once


# grad_input collected in octets of channels: several deformable and convolution groups, halves of octets (the 4-channel chunks of stride 2, and, beside whole
# ones, of wide halos), the path without LDS tiling behind it, and a weight gradient that 16-bit storage computes on widened tensors in the same workspace
OCTETS = [(3, 2, 24, 20, (5, 9, 10), 3, 1, 1, 1, 8, 1, 1.5), (3, 1, 16, 12, (4, 8, 9), 3, 1, 1, 1, 16, 2, 3.5), (3, 1, 16, 33, (9, 21, 19), 3, 2, 1, 1, 16, 1, 2.0),
          (3, 2, 8, 16, (6, 9, 9), 3, 1, 1, 1, 8, 1, 12.0), (3, 1, 64, 128, (4, 9, 10), 3, 1, 1, 1, 32, 1, 1.5), (3, 2, 16, 12, (8, 17, 19), 3, 1, 1, 1, 16, 1, 3.3)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("spec", OCTETS, ids=lambda s: "%d-%d-cpg%d-reach%g" % (s[2], s[3], s[9], s[11]))
def test_octets(spec, dtype):
    """Every gradient of a layer in one call; the same call with grad_input alone wanted besides grad_offset.  Bounds as in test_edges; grad_weight in
    bfloat16: its samples are rounded too."""
    import deform_conv3d_pytorch_op_amd as dcn
    print("octets", spec, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=38, bias=False)
    x, off, w = (c[k].cuda().requires_grad_() for k in ("x", "off", "w"))
    dcn.ConvOffset3dFunction.apply(x, off, w, None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"]).backward(c["gout"].cuda())
    d = {k: c[k].float() for k in ("x", "off", "w", "gout")}
    want = [t.double() for t in orc.backward(d["x"], d["off"], d["w"], d["gout"], None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])[:3]]
    once = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -9}[dtype]
    got = [t.grad.cpu().double() for t in (x, off, w)] + list(_gradients(c))
    for g, t, tol in zip(got, want + want[:2], (1e-4, 1e-5, 1e-5 + 2 * once, 1e-4, 1e-5)):
        err = ((g - t).norm() / t.norm()).item()
        print("  relative 2-norm error %.2e" % err, flush=True)
        assert err <= tol + once


def test_octets_are_taken():
    """What the layers above are for (the trace of the plans, in a process of its own: the knob is read once)."""
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", __file__, "-q", "-x", "-s", "-m", "gpu", "-k", "test_octets and not taken and not behind", "--timeout", "120",
                        "--timeout-method", "thread"], cwd=os.path.dirname(here), env=dict(os.environ, DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    cases = r.stdout.split("octets (")[1:]
    assert len(cases) == 2 * len(OCTETS)
    for case in cases:
        what = case[:case.index("\n")]
        spec, f32 = ast.literal_eval("(" + what[:what.rindex(")") + 1]), what.endswith("torch.float32")
        collected = re.findall(r"grad_input collected in (.*)", case)
        chunks = set(re.findall(r"dcn backward_input_offset: launch.* (\d+) channels per chunk, ", case))
        print(spec, what, collected, chunks, flush=True)
        assert collected and set(collected) == {"octets"}, spec
        assert chunks == ({"4"} if spec == OCTETS[2] else {"8", "4"} if spec == OCTETS[5] else {"8"}), spec
        assert ("grad_input rounded ahead" in case) == (spec == OCTETS[4] and not f32), spec
        assert ("path without LDS tiling offered" in case) == f32, spec


def test_octets_behind_the_path_without_lds():
    """The device takes the path without LDS tiling for the layer of far offsets (the plan is recorded in the workspace, include/dcn_amd.h), whose channels-last
    gradients the octets' last launch then adds to what grad_input holds."""
    from deform_conv3d_pytorch_op_amd import _lib
    from deform_conv3d_pytorch_op_amd.functions import _geom, _workspace_bytes
    print("octets, global", flush=True)
    L, c = _lib.load(), make_case(*OCTETS[3], dtype=torch.float32, seed=38, bias=False)
    x, off, w, gout = (c[k].cuda() for k in ("x", "off", "w", "gout"))
    nbytes = _workspace_bytes(x, w, c["groups"], c["outs"], c["cpg"])
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
    gin, goff = torch.ones_like(x), torch.empty_like(off)
    geom = _geom(3, x, w, c["outs"], c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    assert L.dcn3d_backward_input_offset_f32(*(t.data_ptr() for t in (x, w, off, gout, gin, goff)), *geom, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    at = (nbytes - 256) // 256 * 256 + 64
    assert int.from_bytes(bytes(ws[at:at + 4].cpu().tolist()), "little") == 3
    for got, want, tol in zip((gin - 1, goff), _oracle(c), (1e-4, 1e-5)):
        assert ((got.cpu().double() - want).norm() / want.norm()).item() <= tol


def test_one_small_position_beside_ordinary_ones():
    """grad_offset of positions whose grad_output alone is tiny."""
    print("small position", flush=True)
    c = make_case(2, 1, 16, 48, (24, 40), 3, 1, 1, 1, 16, 1, 0.9, dtype=torch.float32, seed=33, bias=False)
    c["gout"][..., 20:] *= 2.0 ** -119
    got, want = _gradients(c)[1], _oracle(c)[1]
    for part in (slice(0, 20), slice(20, None)):
        g, w = got[..., part], want[..., part]
        assert ((g - w).norm() / w.norm()).item() <= 1e-5


def test_values_whose_parts_round_to_infinity():
    """Weights just below the largest float with gradients that stay finite."""
    print("huge", flush=True)
    c = make_case(3, 1, 12, 20, (4, 9, 9), 3, 1, 1, 1, 12, 1, 1.5, dtype=torch.float32, seed=34, bias=False)
    c["w"].view(-1)[::5] = 3.395e38
    c["gout"] *= 1e-6
    for got, want in zip(_gradients(c), _oracle(c)):
        assert torch.isfinite(want).all()
        assert ((got - want).norm() / want.norm()).item() <= 1e-4
