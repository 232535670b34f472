"""16-bit storage at the edges of what the 16-bit kernels serve themselves: layers whose halo just fits a block
of 256 positions or whose positions are too few to share their columns, layers past that halo, which run the float32
operator on widened tensors, and values that are not finite."""
import pytest
import torch

from oracle import dcn_oracle as orc
from tests.cases import make_case
from tests.test_gpu_mixed import _compare

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
# half a unit in the last place, relative to the value
ROUNDING = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}

# (nd, N, C_in, C_out, ins, k, stride, pad, dil, cpg, groups, reach)
FITS = [(3, 1, 16, 24, (9, 21, 22), 3, 2, 1, 1, 8, 1, 1.5), (3, 2, 12, 40, (6, 17, 18), 3, 1, 3, 3, 12, 1, 1.5), (3, 1, 8, 16, (5, 19, 20), 3, (1, 2, 2), 2, 2, 8, 1, 1.5),
        (2, 1, 24, 72, (70, 62), 5, 3, 6, 3, 24, 1, 2.0), (2, 1, 256, 96, (30, 27), 3, 1, 1, 1, 64, 1, 1.5), (2, 1, 48, 264, (21, 90), 3, 1, 1, 1, 48, 1, 2.0),
        (2, 2, 16, 130, (30, 33), 3, 2, 2, 2, 16, 2, 2.0)]
PAST = [(3, 1, 16, 32, (20, 30, 30), 3, 2, 2, 2, 16, 1, 1.5), (3, 1, 24, 72, (9, 16, 17), 3, 1, 4, 4, 12, 1, 1.5),
        (2, 1, 16, 48, (60, 50), 5, 4, 8, 4, 16, 1, 2.0), (2, 1, 32, 96, (60, 60), 5, 4, 8, 4, 32, 1, 2.0)]


def _forward(c):
    import deform_conv3d_pytorch_op_amd as dcn
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    x, off, w, b = (c[k].cuda() for k in ("x", "off", "w", "b"))
    return fn.apply(x, off, w, b, c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"]).cpu()


def _id(s):
    return "%dd-%d-%d-k%s-s%s-d%s" % (s[0], s[2], s[3], s[5], s[6], s[8])


@pytest.mark.parametrize("dtype", DTYPES.values(), ids=DTYPES)
@pytest.mark.parametrize("spec", FITS, ids=_id)
def test_layers_that_fit(spec, dtype):
    print("fits", spec, dtype, flush=True)
    _compare(make_case(*spec, dtype=dtype, seed=41), dtype, "fits")


@pytest.mark.parametrize("dtype", DTYPES.values(), ids=DTYPES)
@pytest.mark.parametrize("spec", PAST, ids=_id)
def test_layers_past_the_halo_keep_float32_samples(spec, dtype):
    """The float32 result rounded once: no more than half a unit of the last place away from it, plus what the
    order of float32 sums changes."""
    print("past", spec, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=42)
    got = _forward(c).float()
    want = _forward({k: v.float() if torch.is_tensor(v) else v for k, v in c.items()})
    assert bool(((got - want).abs() <= ROUNDING[dtype] * want.abs() + 2e-6 * want.abs().max()).all())


@pytest.mark.parametrize("dtype", DTYPES.values(), ids=DTYPES)
@pytest.mark.parametrize("what", ["x", "w"])
@pytest.mark.parametrize("spec", [(2, 1, 20, 65, (19, 33), 3, 1, 1, 1, 20, 1, 1.5), (2, 1, 40, 257, (16, 33), 3, 1, 1, 1, 40, 1, 1.0),
                                  (3, 1, 12, 64, (5, 9, 10), 3, 1, 1, 1, 4, 1, 1.5)], ids=["2d", "2d-wide", "3d"])
def test_results_that_are_not_finite(spec, what, dtype):
    """Infinities keep their sign and NaN stay, in exactly the results that the reference's arithmetic gives them."""
    print("not finite", spec, what, dtype, flush=True)
    c = make_case(*spec, dtype=dtype, seed=43)
    t = c[what].view(-1)
    t[torch.randperm(t.numel(), generator=torch.Generator().manual_seed(4))[:3]] = torch.tensor([float("inf"), -float("inf"), float("nan")], dtype=dtype)
    d = {k: c[k].float() for k in ("x", "off", "w", "b")}
    got, want = _forward(c).float(), orc.forward(d["x"], d["off"], d["w"], d["b"], c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"])
    for special in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(special(got), special(want))
    fin = torch.isfinite(want)
    assert fin.any() and not fin.all()
    assert (got - want)[fin].abs().max().item() <= (5e-3 if dtype == torch.bfloat16 else 1e-3) * want[fin].abs().max().item()
