"""The allocation-free entry point at the largest weights it accepts: deformable groups of four channels, whose
packed weights take three times the accepted size, still run on the LDS-halo kernel."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SCRIPT = """
import torch
from deform_conv3d_pytorch_op_amd import _lib
from tests.test_zz_no_alloc import _both
got, want = _both(_lib.load(), (1, 144, 256, (3, 6, 7), 3, 1, 1, 1, 4, 1, 1.5), seed=13, poison=7.0)
err = ((got - want).abs().max() / want.abs().max()).item()
print("relative error %.3e" % err, flush=True)
assert err <= 1e-6
"""


def test_largest_accepted_layer_runs_on_the_halo_kernel():
    print("no-alloc limit", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", SCRIPT], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       env=dict(os.environ, DCN_TRACE_PLANS="1"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-3000:]
    assert r.stdout.count("dcn forward:") == 3, r.stdout[-3000:]        # dcn3d_forward_f32 once, the allocation-free call twice
