"""The halo plans of the forward pass's 1024-thread shape: layers large enough for it, offsets for each margin that the
device chooses among and beyond the widest one."""
import pytest
import torch

from oracle import dcn_oracle as orc
from tests.cases import make_case

pytestmark = pytest.mark.gpu

# 3-D, 20 channels per pass or fewer (eight, then four, as the halo widens); 2-D
LAYERS = {"3d": (3, 3, 20, 33, (17, 55, 57), 3, 1, 1, 1, 20, 1), "2d": (2, 8, 24, 40, (131, 150), 3, 1, 1, 1, 24, 1)}


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.bfloat16, 4e-3)], ids=["f32", "bf16"])
@pytest.mark.parametrize("reach", [1.9, 2.9, 3.9, 5.9, 8.0])
@pytest.mark.parametrize("name", LAYERS)
def test_wide_offsets(name, reach, dtype, tol):
    """2-norm error against the oracle in float32 coordinates and float64 sums (bfloat16: samples rounded once, 2^-9, and
    the result once)."""
    import deform_conv3d_pytorch_op_amd as dcn
    print("halo plans", name, reach, dtype, flush=True)
    c = make_case(*LAYERS[name], reach, dtype=dtype, seed=51)
    cfg = (c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    got = fn.apply(*(c[k].cuda() for k in ("x", "off", "w", "b")), *cfg).cpu().double()
    want = orc.forward(*(c[k].float() for k in ("x", "off", "w", "b")), *cfg).double()
    err = ((got - want).norm() / want.norm()).item()
    print("  relative 2-norm error %.2e" % err, flush=True)
    assert err <= tol
