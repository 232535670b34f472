"""The forward pass with eight and sixteen wavefronts to a position: edges of its blocks, its parts of the input channels,
and the shape with four wavefronts that it took over from."""
import os
import re
import subprocess
import sys

import pytest
import torch

from tests.cases import make_case
from tests.test_gpu_split import _forward, _oracle

pytestmark = pytest.mark.gpu

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): blocks of 32 positions and their remainders, of 64 where
# those of 32 are more than 256; one and two row tiles; one tap; channel parts that fall unevenly; wide offsets.  The rule's estimate
# leaves some of them to four wavefronts to a position: test_forced_shapes runs all of them on blocks of 32 and of 64.  (5x5 on 95 x 97 at
# padding 1: at padding 2 one coordinate rounds onto the border in float32 and not in the oracle's float64, which drops a sample, 1.6e-3.)
EDGES = [
    (2, 1, 8, 1, (5, 5), 3, 1, 1, 1, 8, 1, 1.0), (2, 1, 20, 33, (4, 33), 3, 1, 1, 1, 20, 1, 1.5), (2, 1, 160, 64, (9, 8), 3, 1, 1, 1, 80, 1, 2.0),
    (2, 2, 24, 40, (31, 30), 1, 1, 0, 1, 12, 1, 2.0), (2, 1, 16, 32, (100, 101), 3, 1, 1, 1, 16, 1, 3.5), (2, 1, 40, 48, (130, 128), 5, 2, 2, 1, 20, 2, 1.5),
    (3, 1, 8, 32, (3, 4, 5), 3, 1, 1, 1, 8, 1, 1.5), (3, 1, 48, 64, (5, 9, 9), 3, 1, 1, 1, 24, 1, 2.5), (3, 2, 12, 20, (9, 19, 23), 3, 1, 1, 1, 4, 1, 1.5),
    (3, 1, 64, 34, (6, 10, 11), 2, 2, 1, 1, 32, 2, 7.0), (2, 1, 256, 40, (31, 30), 1, 1, 0, 1, 128, 1, 2.0), (2, 1, 64, 64, (100, 101), 3, 1, 1, 1, 64, 1, 1.5),
    (2, 1, 96, 33, (95, 97), 5, 1, 1, 1, 48, 1, 2.0), (2, 1, 160, 30, (99, 90), 3, 1, 1, 1, 160, 1, 2.0), (3, 1, 48, 50, (9, 30, 35), 3, 1, 1, 1, 48, 1, 1.5),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("spec", EDGES, ids=lambda s: "%dd-%d-%d-k%d-cpg%d" % (s[0], s[2], s[3], s[5], s[9]))
def test_edges(spec, dtype):
    """2-norm: a chain of float32 roundings (2e-6) and a coordinate rounded by up to 2^-18 (half a unit below 128), which moves a sample
    of N(0, 1) values by as much; 16-bit storage rounds the samples and the results once (2^-9 and 2^-12 of each), and an offset beside
    an integer may sample the other side of a corner in float64."""
    print("edges", spec, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=41)
    got, want = _forward(c).cpu().double(), _oracle(c)
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= {torch.float32: 2e-6 + 2.0 ** -18, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]


def _rerun(knobs, files, k):
    """The output of a process of its own (the knobs are read once) that runs the tests `k` of these files."""
    print("knobs", knobs, flush=True)
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", *(os.path.join(here, f) for f in files), "-q", "-x", "-s", "-m", "gpu", "-k", k,
                        "--timeout", "120", "--timeout-method", "thread"],
                       cwd=os.path.dirname(here), env=dict(os.environ, **knobs), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    return r.stdout


def _shapes(trace):
    """Of every case of test_edges that the trace of the plans holds: storage type, (position tiles of a block, wavefronts, row tiles)."""
    return [(re.search(r"torch\.(\w+)", case).group(1),
             tuple(int(m) for m in re.search(r"dcn forward: (\d+) position tiles, (\d+) wavefronts, MT (\d+)", case).groups()))
            for case in trace.split("edges (")[1:]]


def test_shapes_of_the_rule():
    """What the rule makes of the cases above: in every storage type both blocks, with one and with two row tiles, and four wavefronts."""
    shapes = _shapes(_rerun({"DCN_TRACE_PLANS": "1"}, ["test_gpu_tiny.py"], "test_edges"))
    print(shapes, flush=True)
    assert len(shapes) == 3 * len(EDGES)
    for dtype in ("float32", "bfloat16", "float16"):
        for want in ((1, 16, 1), (1, 16, 2), (2, 16, 1), (2, 16, 2), (2, 8, 1)):
            assert (dtype, want) in shapes, (dtype, want)


@pytest.mark.parametrize("tiles", [1, 2])
def test_forced_shapes(tiles):
    """Every case above on blocks of 32 positions with sixteen wavefronts to a position, and of 64 with eight."""
    shapes = _shapes(_rerun({"DCN_FORWARD_TINY": str(tiles), "DCN_TRACE_PLANS": "1"}, ["test_gpu_tiny.py"], "test_edges"))
    print(shapes, flush=True)
    assert len(shapes) == 3 * len(EDGES) and {s for _, s in shapes} == {(tiles, 16, 1), (tiles, 16, 2)}


@pytest.mark.parametrize("knobs", [{"DCN_FORWARD_TINY": "0"}, {"DCN_FORWARD_TINY": "1"}, {"DCN_FORWARD_TINY": "2"}, {"DCN_FORWARD_SPLIT": "1"}],
                         ids=["four-wavefronts", "sixteen", "eight", "no-parts"])
def test_other_shapes(knobs):
    """The same layers with four, sixteen and eight wavefronts to a position, and in one part."""
    _rerun(knobs, ["test_gpu_tiny.py", "test_gpu_split.py", "test_gpu_parity.py"],
           "(edges or not_finite or small_cases) and not larger_shapes and not other_shapes")
