"""backward_weight_split_kernel: layers just large enough for it, with the edges of its tiles, slabs, segments and volumes."""
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

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): two and four row tiles and their remainders, one and
# several chunks of them; channel tiles with remainders; deformable groups over two convolution groups; last slabs of 1 and 31
# positions and whole ones; strides and dilations; an axis of one voxel; one tap of many channels; samples past the volume
LAYERS = [
    (2, 1, 33, 65, (97, 161), 3, 1, 1, 1, 33, 1, 1.5), (2, 2, 40, 128, (97, 73), 3, 1, 1, 1, 20, 1, 3.0),
    (2, 1, 24, 210, (141, 99), 3, 1, 1, 1, 8, 2, 2.0), (2, 3, 33, 33, (85, 89), 3, 1, 1, 1, 33, 1, 1.0),
    (2, 1, 32, 64, (229, 231), 5, 2, 2, 1, 32, 1, 9.0), (2, 1, 136, 97, (221, 223), 1, 1, 0, 1, 136, 1, 0.9),
    (3, 1, 16, 80, (9, 32, 32), 3, 1, 1, 1, 16, 1, 1.5), (3, 2, 5, 66, (13, 39, 41), 3, (1, 2, 2), 1, 1, 5, 1, 2.5),
    (3, 1, 34, 40, (1, 95, 97), 3, 1, 1, 1, 17, 1, 1.0), (3, 1, 12, 70, (23, 21, 25), 3, 1, 2, 2, 12, 2, 2.0),
    # two and four taps to an item (segments of up to 16 and 8 channels), up to 32 output channels too
    (2, 1, 16, 65, (161, 163), 3, 1, 1, 1, 16, 1, 1.5), (2, 2, 42, 130, (97, 73), 3, 1, 1, 1, 14, 1, 3.0), (2, 1, 48, 40, (145, 147), 3, 1, 1, 1, 48, 1, 1.0),
    (2, 1, 15, 20, (257, 259), 3, 2, 1, 1, 5, 1, 2.0), (2, 1, 8, 34, (229, 231), 5, 2, 2, 1, 8, 1, 9.0), (3, 1, 16, 20, (11, 32, 33), 3, 1, 1, 1, 4, 2, 1.5),
    (3, 1, 7, 66, (13, 39, 41), 3, 1, 1, 1, 7, 1, 2.5), (3, 1, 16, 33, (17, 33, 35), 3, 1, 1, 1, 16, 1, 2.5), (3, 1, 12, 40, (1, 131, 133), 3, 1, 1, 1, 3, 1, 1.0),
    # eight row tiles (129 to 256 output channels to a group): their least and their most, two groups; nine tiles take chunks of four
    (2, 1, 33, 129, (97, 101), 3, 1, 1, 1, 33, 1, 1.5), (2, 1, 40, 256, (97, 97), 3, 1, 1, 1, 40, 1, 2.5), (2, 1, 40, 420, (101, 99), 3, 1, 1, 1, 20, 2, 9.0),
    (3, 1, 33, 161, (9, 21, 35), 3, 1, 1, 1, 33, 1, 1.5), (2, 1, 160, 250, (223, 225), 1, 1, 0, 1, 160, 1, 0.9), (2, 1, 33, 288, (97, 101), 3, 1, 1, 1, 33, 1, 1.5),
    # 16 bytes of a corner to a lane: segments that end one lane into a tile, also two and four taps to an item; one over two convolution groups
    (2, 1, 36, 70, (97, 161), 3, 1, 1, 1, 36, 1, 1.5), (2, 1, 40, 130, (161, 99), 3, 1, 1, 1, 40, 2, 3.0), (2, 1, 12, 65, (161, 163), 3, 1, 1, 1, 12, 1, 9.0),
    (2, 1, 4, 66, (229, 231), 3, 1, 1, 1, 4, 1, 1.5), (2, 1, 68, 66, (1, 9001), 3, 1, 1, 1, 68, 1, 1.5),
    # slabs of four octets apart, 3-D: rows of several octets with slabs left over, rows shorter than an octet, two samples
    (3, 1, 17, 66, (3, 41, 75), 3, 1, 1, 1, 17, 1, 1.5), (3, 1, 9, 70, (203, 16, 3), 3, 1, 1, 1, 9, 1, 1.5), (3, 2, 16, 129, (5, 31, 47), 3, 1, 1, 1, 16, 1, 9.0),
]
# (row tiles, lanes to a tap, bytes of a corner to a lane) of layers whose variant is one of few: eight row tiles, 16 bytes to a lane with 32, 16 and 8 lanes
VARIANTS = {
    (2, 1, 33, 129, (97, 101), 3, 1, 1, 1, 33, 1, 1.5): (8, 32, 4), (2, 1, 40, 256, (193, 195), 3, 1, 1, 1, 40, 1, 2.5): (8, 32, 16),
    (2, 1, 40, 420, (131, 133), 3, 1, 1, 1, 20, 2, 9.0): (8, 32, 16), (3, 1, 33, 161, (9, 21, 35), 3, 1, 1, 1, 33, 1, 1.5): (8, 32, 4),
    (2, 1, 160, 250, (223, 225), 1, 1, 0, 1, 160, 1, 0.9): (8, 32, 16), (2, 1, 36, 70, (97, 161), 3, 1, 1, 1, 36, 1, 1.5): (4, 32, 16),
    (2, 1, 68, 66, (1, 9301), 3, 1, 1, 1, 68, 1, 1.5): (4, 32, 16), (2, 1, 32, 65, (161, 163), 3, 1, 1, 1, 16, 1, 1.5): (4, 16, 16),
    (2, 1, 24, 65, (161, 163), 3, 1, 1, 1, 12, 1, 9.0): (4, 16, 16), (2, 1, 16, 66, (161, 163), 3, 1, 1, 1, 8, 1, 1.5): (4, 8, 16),
    (2, 1, 16, 40, (161, 163), 3, 1, 1, 1, 4, 1, 1.5): (2, 8, 16), (2, 1, 33, 65, (97, 161), 3, 1, 1, 1, 33, 1, 1.5): (4, 32, 4),
    (3, 1, 17, 66, (3, 41, 75), 3, 1, 1, 1, 17, 1, 1.5): (4, 32, 4),
}
LAYERS += [s for s in VARIANTS if s not in LAYERS]
IDS = lambda s: "%dd-%d-%d-k%d-g%d" % (s[0], s[2], s[3], s[5], s[10])


def _weight_gradient(c):
    import deform_conv3d_pytorch_op_amd as dcn
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    x, off, w = (c[k].cuda().requires_grad_(k == "w") for k in ("x", "off", "w"))
    b = torch.zeros(w.shape[0], device="cuda", dtype=w.dtype).requires_grad_(True)
    fn.apply(x, off, w, b, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"]).backward(c["gout"].cuda())
    return w.grad.cpu().double(), b.grad.cpu().double()


def _oracle(c):
    """In float32 with double sums: the coordinates are then those of the kernel."""
    d = {k: c[k].float() for k in ("x", "off", "w", "gout")}
    return orc.backward(d["x"], d["off"], d["w"], d["gout"], None, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])[2].double()


@pytest.mark.parametrize("spec", LAYERS, ids=IDS)
def test_layers(spec):
    """2-norm: chains of float32 sums over up to a few hundred steps of positions and the splits, each off by half a unit in
    the last place of a partial sum: below 2^-24 * 64 = 4e-6."""
    print("weight gradient", spec, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=41, bias=False)
    got, bias = _weight_gradient(c)
    want = _oracle(c)
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= 4e-6
    g64 = c["gout"].double()
    sums = g64.sum(dim=[0] + list(range(2, g64.dim())))
    assert ((bias - sums).norm() / sums.norm()).item() <= 4e-6


# 16-bit storage: pairs of channels, so even segments
LAYERS16 = [
    (2, 1, 34, 70, (129, 161), 3, 1, 1, 1, 34, 1, 1.5), (2, 2, 66, 40, (129, 161), 3, 1, 1, 1, 66, 1, 3.0),
    (2, 1, 24, 120, (141, 99), 3, 1, 1, 1, 8, 2, 2.0), (3, 1, 20, 64, (9, 32, 33), 3, 1, 1, 1, 10, 1, 1.5),
    (3, 1, 40, 97, (7, 31, 32), 3, 1, 1, 1, 40, 1, 2.5), (3, 1, 2, 60, (1, 95, 97), 3, 1, 1, 1, 2, 1, 1.0),
    (3, 1, 16, 30, (17, 33, 35), 3, 1, 1, 1, 16, 1, 2.5), (2, 1, 60, 64, (129, 161), 3, 1, 1, 1, 30, 1, 1.5), (2, 1, 24, 66, (129, 161), 3, 1, 1, 1, 24, 1, 1.5),
    (2, 1, 72, 70, (129, 161), 3, 1, 1, 1, 72, 1, 1.5), (3, 1, 48, 64, (7, 31, 33), 3, 1, 1, 1, 24, 1, 2.5), (3, 1, 80, 64, (1, 95, 97), 3, 1, 1, 1, 80, 2, 1.0),
    (2, 1, 16, 130, (129, 161), 3, 1, 1, 1, 16, 1, 9.0), (2, 1, 8, 66, (229, 231), 3, 1, 1, 1, 8, 1, 1.5),
]
# ... of the kernel that reads 16-bit storage; where two are given, bfloat16's and binary16's
VARIANTS16 = {
    (2, 1, 72, 64, (129, 161), 3, 1, 1, 1, 72, 1, 1.5): (2, 32, 16), (3, 1, 40, 97, (7, 31, 32), 3, 1, 1, 1, 40, 1, 2.5): (4, 32, 16),
    (3, 1, 160, 128, (1, 95, 97), 3, 1, 1, 1, 160, 2, 1.0): (2, 32, 16), (3, 1, 48, 64, (7, 31, 33), 3, 1, 1, 1, 24, 1, 2.5): (2, 16, 16),
    (2, 1, 32, 64, (129, 161), 3, 1, 1, 1, 16, 1, 9.0): (2, 8, 16), (2, 1, 16, 40, (161, 163), 3, 1, 1, 1, 8, 1, 1.5): (2, 8, 16),
    (3, 1, 32, 64, (9, 32, 33), 3, 1, 1, 1, 16, 1, 1.5): ((2, 8, 4), (2, 8, 16)), (3, 1, 16, 30, (17, 33, 35), 3, 1, 1, 1, 16, 1, 2.5): (1, 8, 16),
}
LAYERS16 += [s for s in VARIANTS16 if s not in LAYERS16]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("spec", LAYERS16, ids=IDS)
def test_layers_16bit(spec, dtype):
    """Samples and results are rounded to the storage format, each off by half a unit in its last place at most: 2-norm
    below 2^-9 and 2^-12 each.  Non-finite input reaches the elements that it reaches in the oracle."""
    print("weight gradient", spec, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=45, bias=False)
    got, bias = _weight_gradient(c)
    want = _oracle(c)
    once = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    assert ((got - want).norm() / want.norm()).item() <= 2 * once
    g64 = c["gout"].double()
    sums = g64.sum(dim=[0] + list(range(2, g64.dim())))
    assert ((bias - sums).norm() / sums.norm()).item() <= once + 4e-6
    c["x"][0, -1].view(-1)[-3:] = torch.tensor([float("inf"), float("nan"), -float("inf")])
    got, _ = _weight_gradient(c)
    want = _oracle(c)
    fin = torch.isfinite(want)
    assert not fin.all() and torch.equal(torch.isfinite(got), fin)
    assert ((got - want)[fin].norm() / want[fin].norm()).item() <= 2 * once


EXACT = [LAYERS[0], LAYERS[6]] + [s for s in VARIANTS if s[3] in (129, 256) or s[2:4] in ((36, 70), (24, 65))]


def test_variants_of_the_layers():
    """The layers take the variants that they are here for (the trace of the plans, in a process of its own: the knob is read once)."""
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", __file__, "-q", "-x", "-s", "-m", "gpu", "-k", "test_layers", "--timeout", "120", "--timeout-method", "thread"],
                       cwd=os.path.dirname(here), env=dict(os.environ, DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    seen = 0
    for case in r.stdout.split("weight gradient (")[1:]:
        what = case[:case.index("\n")]
        spec, dtype = ast.literal_eval("(" + what[:what.rindex(")") + 1]), what[what.rindex(")") + 1:].strip() or "torch.float32"
        want = (VARIANTS if dtype == "torch.float32" else VARIANTS16).get(spec)
        if want is None:
            continue
        if isinstance(want[0], tuple):
            want = want[dtype == "torch.float16"]
        got = re.findall(r"dcn backward_weight, (\w+): (\d+) row tiles, (\d+) lanes to a tap, (\d+) bytes", case)
        print(spec, dtype, got, flush=True)
        storage = {"torch.float32": "float32", "torch.bfloat16": "bfloat16", "torch.float16": "binary16"}[dtype]
        assert got and set(got) == {(storage,) + tuple(map(str, want))}, spec
        seen += 1
    assert seen == len(VARIANTS) + 2 * len(VARIANTS16)


@pytest.mark.parametrize("spec", EXACT, ids=IDS)
@pytest.mark.parametrize("what,exponent", [("gout", 90), ("gout", 120), ("x", 100), ("x", 126)])
def test_small_operands(spec, what, exponent):
    """Operands whose bfloat16 parts leave the range of normal numbers: the results are formed from the values themselves."""
    print("small", spec, what, exponent, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=42, bias=False)
    c[what] = c[what] * 2.0 ** -exponent
    got, _ = _weight_gradient(c)
    want = _oracle(c)
    if exponent >= 120:                 # results and partial sums near the smallest normal number, off by a few of its last units
        assert (got - want).abs().max().item() <= 2.0 ** -149 * 64 + 4e-6 * want.abs().max().item()
    else:
        assert ((got - want).norm() / want.norm()).item() <= 4e-6


@pytest.mark.parametrize("spec", EXACT, ids=IDS)
@pytest.mark.parametrize("what", ["x", "gout", "off"])
def test_non_finite(spec, what):
    """Not finite where the oracle's gradient is not, equal to it elsewhere."""
    print("non-finite", spec, what, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=43, bias=False)
    flat = c[what].view(-1)
    if what == "x":                     # the last channel alone, in the last rows of the volume: the collapsed corners lie there
        c["x"][0, -1].view(-1)[-3:] = torch.tensor([float("inf"), float("nan"), -float("inf")])
    elif what == "gout":
        c["gout"][0, -1].view(-1)[5:8] = torch.tensor([float("inf"), float("nan"), -float("inf")])
    else:
        flat[::997] = float("nan")
        flat[5::1009] = float("inf")
    got, _ = _weight_gradient(c)
    want = _oracle(c)
    fin = torch.isfinite(want)
    assert what == "off" or not fin.all()
    assert torch.equal(torch.isfinite(got), fin)
    assert ((got - want)[fin].norm() / want[fin].norm()).item() <= 4e-6


@pytest.mark.parametrize("n,ci,co,size", [(2, 40, 70, (83, 85)), (4, 33, 64, (73, 91))])
def test_plain_convolution(n, ci, co, size):
    """The convolution without offsets, against float64."""
    import deform_conv3d_pytorch_op_amd as dcn
    print("plain", n, ci, co, size, flush=True)
    g = torch.Generator().manual_seed(44)
    x = torch.randn((n, ci) + size, generator=g)
    m = dcn.Conv2d(ci, co, 3, 1, 1, 1, device="cuda")
    gout = torch.randn((n, co) + size, generator=g)
    m(x.cuda()).backward(gout.cuda())
    want = torch.nn.grad.conv2d_weight(x.double(), m.weight.shape, gout.double(), stride=1, padding=1)
    assert ((m.weight.grad.cpu().double() - want).norm() / want.norm()).item() <= 4e-6
