"""The float32 contraction from bfloat16 parts: edges of its tiles and groups, its accuracy, and the
results that are not finite (worked out on the float32 instructions)."""
import os
import subprocess
import sys

import pytest
import torch

from oracle import dcn_oracle as orc
from tests.cases import make_case

pytestmark = pytest.mark.gpu


def _forward(c):
    import deform_conv3d_pytorch_op_amd as dcn
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    x, off, w = (c[k].cuda() for k in ("x", "off", "w"))
    b = c["b"].cuda() if c["b"] is not None else None
    return fn.apply(x, off, w, b, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])


def _oracle(c):
    d = {k: c[k].double() if c[k] is not None else None for k in ("x", "off", "w", "b")}
    return orc.forward(d["x"], d["off"], d["w"], d["b"], c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])


# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): groups of eight channels and their
# remainders (4, 12, 20 channels; segments of 4), row tiles (32, 33, 64, 65, 129, 257 output channels),
# odd and even tap counts, one tap, samples past every halo
EDGES = [
    (2, 1, 4, 32, (9, 17), 3, 1, 1, 1, 4, 1, 1.0), (2, 2, 12, 33, (12, 12), 3, 1, 1, 1, 12, 1, 2.0),
    (2, 1, 20, 65, (19, 33), 3, 1, 1, 1, 20, 1, 1.5), (2, 1, 24, 129, (17, 16), 2, 1, 0, 1, 12, 1, 2.5),
    (2, 1, 40, 257, (16, 33), 3, 1, 1, 1, 40, 1, 1.0), (2, 1, 16, 160, (11, 11), 1, 1, 0, 1, 4, 2, 1.5),
    (2, 1, 72, 96, (20, 20), 3, 2, 1, 2, 24, 3, 9.0), (3, 1, 12, 64, (5, 9, 10), 3, 1, 1, 1, 4, 1, 1.5),
    (3, 1, 20, 33, (4, 8, 9), 3, 1, 1, 1, 20, 1, 1.0), (3, 1, 8, 130, (6, 9, 9), 2, 1, 1, 1, 8, 1, 6.0),
    (3, 1, 24, 48, (9, 21, 22), 3, 2, 1, 2, 12, 2, 3.0),
]


@pytest.mark.parametrize("spec", EDGES, ids=lambda s: "%dd-%d-%d-k%d-cpg%d" % (s[0], s[2], s[3], s[5], s[9]))
def test_edges_and_accuracy(spec):
    """Error against the float64 oracle in the 2-norm: what a chain of float32 roundings leaves."""
    print("edges", spec, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=21)
    got, want = _forward(c).cpu().double(), _oracle(c)
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= 2e-6


# 3-D layers whose halo of 256 positions holds no eight channels, of more blocks of 64 positions than the device holds at once: few
# input channels and several row tiles, one and two row tiles, groups, samples past every halo, 125 taps
WIDE_HALOS = [(3, 2, 8, 70, (33, 65, 66), 3, 2, 1, 1, 8, 1, 1.5), (3, 1, 32, 20, (41, 66, 67), 3, 2, 1, 1, 16, 1, 2.5), (3, 1, 36, 40, (41, 66, 67), 3, 2, 1, 1, 12, 1, 9.0),
              (3, 1, 64, 140, (35, 50, 51), 3, 2, 1, 1, 64, 2, 1.0), (3, 1, 8, 66, (25, 66, 67), 5, 2, 2, 1, 4, 1, 1.5)]


@pytest.mark.parametrize("spec", WIDE_HALOS, ids=lambda s: "%d-%d-k%d-cpg%d" % (s[2], s[3], s[5], s[9]))
def test_wide_halos(spec):
    """2-norm: a chain of float32 roundings (2e-6) and a coordinate rounded by up to 2^-18 (half a unit below 128), which moves a sample
    of N(0, 1) values by as much."""
    print("wide halos", spec, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=24)
    got, want = _forward(c).cpu().double(), _oracle(c)
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= 2e-6 + 2.0 ** -18


@pytest.mark.parametrize("spec", [EDGES[2], EDGES[4], EDGES[7]], ids=["2d-split", "2d-shared", "3d"])
@pytest.mark.parametrize("what", ["input", "weight", "huge"])
def test_results_that_are_not_finite(spec, what):
    """Infinities keep their sign, NaN stay, and values whose parts would round to infinity do not."""
    print("not finite", spec, what, flush=True)
    c = make_case(*spec, dtype=torch.float32, seed=22)
    if what == "huge":
        c["x"].view(-1)[::7] = 3.395e38        # rounds to infinity in bfloat16
        c["w"].mul_(1e-3)
    else:
        t = c["x" if what == "input" else "w"].view(-1)
        at = torch.randperm(t.numel(), generator=torch.Generator().manual_seed(4))[:3]
        t[at] = torch.tensor([float("inf"), -float("inf"), float("nan")])
    got, want = _forward(c).cpu(), _oracle(c)
    for special in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(special(got), special(want))
    fin = torch.isfinite(want)
    assert fin.any() and (what == "huge" or not fin.all())
    assert ((got - want)[fin].double().norm() / want[fin].double().norm()).item() <= 1e-5


@pytest.mark.parametrize("knob", ["DCN_FORWARD_SMALL", "DCN_FORWARD_SHARED"])
def test_larger_shapes_of_the_kernels(knob):
    """Layers this small are worked on by several wavefronts to a position, and wide ones share their
    columns: the same layers through the shapes that larger ones take (one process per setting: the
    knobs are read once)."""
    print("knob", knob, flush=True)
    env = dict(os.environ, **{knob: "0"})
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", __file__, os.path.join(os.path.dirname(__file__), "test_gpu_parity.py"),
                        "-q", "-x", "-m", "gpu", "-k", "(edges or not_finite or small_cases or random_medium) and f32 or edges or not_finite",
                        "--timeout", "120", "--timeout-method", "thread"],
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
