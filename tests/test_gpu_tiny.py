"""The forward pass with eight and sixteen wavefronts to a position: edges of its blocks, its parts of the input channels,
and the shape with four wavefronts that it took over from."""
import os
import subprocess
import sys

import pytest
import torch

from tests.cases import make_case
from tests.test_gpu_split import _forward, _oracle

pytestmark = pytest.mark.gpu

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): blocks of 32 positions and their remainders, of 64 where
# those of 32 are more than 256; one and two row tiles; one tap; channel parts that fall unevenly; wide offsets
EDGES = [
    (2, 1, 8, 1, (5, 5), 3, 1, 1, 1, 8, 1, 1.0), (2, 1, 20, 33, (4, 33), 3, 1, 1, 1, 20, 1, 1.5), (2, 1, 160, 64, (9, 8), 3, 1, 1, 1, 80, 1, 2.0),
    (2, 2, 24, 40, (31, 30), 1, 1, 0, 1, 12, 1, 2.0), (2, 1, 16, 32, (100, 101), 3, 1, 1, 1, 16, 1, 3.5), (2, 1, 40, 48, (130, 128), 5, 2, 2, 1, 20, 2, 1.5),
    (3, 1, 8, 32, (3, 4, 5), 3, 1, 1, 1, 8, 1, 1.5), (3, 1, 48, 64, (5, 9, 9), 3, 1, 1, 1, 24, 1, 2.5), (3, 2, 12, 20, (9, 19, 23), 3, 1, 1, 1, 4, 1, 1.5),
    (3, 1, 64, 34, (6, 10, 11), 2, 2, 1, 1, 32, 2, 7.0),
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


@pytest.mark.parametrize("knobs", [{"DCN_FORWARD_TINY": "0"}, {"DCN_FORWARD_SPLIT": "1"}], ids=["four-wavefronts", "no-parts"])
def test_other_shapes(knobs):
    """The same layers with four wavefronts to a position, and in one part (one process per setting: the knobs are read once)."""
    print("knobs", knobs, flush=True)
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-u", "-m", "pytest", __file__, os.path.join(here, "test_gpu_split.py"), os.path.join(here, "test_gpu_parity.py"),
                        "-q", "-x", "-m", "gpu", "-k", "(edges or not_finite or small_cases) and not larger_shapes and not other_shapes",
                        "--timeout", "120", "--timeout-method", "thread"],
                       cwd=os.path.dirname(here), env=dict(os.environ, **knobs), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
