"""The one-call backward pass (dcn_layer_backward): every set of wanted gradients, against the oracle, at sizes
around the strips and tiles of its preparing launch."""
import pytest
import torch

from oracle import dcn_oracle as orc
from tests.cases import make_case

pytestmark = pytest.mark.gpu

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach): one voxel strip and several, channels
# around a tile of 32, one position, many samples
SPECS = [(2, 3, 5, 33, (3, 5), 3, 1, 1, 1, 5, 1, 1.0), (2, 1, 32, 31, (16, 16), 3, 1, 1, 1, 16, 1, 1.0),
         (2, 2, 34, 66, (17, 31), 3, 1, 1, 1, 34, 2, 2.0), (3, 1, 8, 6, (3, 9, 11), 3, 1, 1, 1, 4, 2, 1.5),
         (3, 5, 4, 8, (2, 3, 2), 1, 1, 0, 1, 4, 1, 0.9)]
WANTED = ["x", "off", "w", "b", "wb", "xb", "xw", "xoffwb"]
TOL = {torch.float32: 1e-4, torch.float64: 1e-10, torch.bfloat16: 2e-2}


@pytest.mark.parametrize("dtype", list(TOL), ids=["f32", "f64", "bf16"])
@pytest.mark.parametrize("spec", SPECS, ids=lambda s: "%dd-n%d-%d-%d" % (s[0], s[1], s[2], s[3]))
def test_wanted_gradients(spec, dtype):
    import deform_conv3d_pytorch_op_amd as dcn
    c = make_case(*spec, dtype=torch.float64, seed=31)
    c = {k: v.to(dtype) if torch.is_tensor(v) else v for k, v in c.items()}
    d = {k: c[k].double() for k in ("x", "off", "w", "b", "gout")}
    cfg = (c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    want = dict(zip(("x", "off", "w", "b"), orc.backward(d["x"], d["off"], d["w"], d["gout"], d["b"], *cfg)))
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    for wanted in WANTED:
        print("wanted", spec, dtype, wanted, flush=True)
        names = [n for n in ("x", "off", "w", "b") if n in wanted.replace("off", "") or (n == "off" and "off" in wanted)]
        t = {n: c[n].cuda().requires_grad_(n in names) for n in ("x", "off", "w", "b")}
        fn.apply(t["x"], t["off"], t["w"], t["b"], *cfg).backward(c["gout"].cuda())
        for n in t:
            if n not in names:
                assert t[n].grad is None
                continue
            err = (t[n].grad.cpu().double() - want[n]).norm() / want[n].norm().clamp_min(1e-30)
            assert err.item() <= TOL[dtype], (wanted, n, err.item())
