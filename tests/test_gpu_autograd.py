"""The package's Functions beside backward: derived classes, tracing, forward mode, saved-tensor hooks,
undefined and misshapen gradients."""
import pytest
import torch

from tests.cases import make_case

pytestmark = pytest.mark.gpu

LAYERS = {"2d": (2, 1, 8, 6, (7, 9), 3, 1, 1, 1, 4, 2, 1.5), "3d": (3, 1, 4, 6, (4, 5, 6), 3, 1, 1, 1, 4, 1, 1.5), "conv2d": None}


def _layer(name):
    """The Function, its arguments (leaves on the GPU that need gradients first) and a grad_output."""
    import deform_conv3d_pytorch_op_amd as dcn
    if name == "conv2d":
        g = torch.Generator().manual_seed(5)
        leaves = [torch.randn(s, generator=g).cuda().requires_grad_() for s in ((2, 6, 8, 7), (4, 3, 3, 3), (4,))]
        return dcn.Conv2dFunction, leaves, ((1, 1), (1, 1), (1, 1), 2), torch.randn((2, 4, 8, 7), generator=g).cuda()
    c = make_case(*LAYERS[name], dtype=torch.float32, seed=5)
    fn = dcn.ConvOffset3dFunction if c["nd"] == 3 else dcn.ConvOffset2dFunction
    leaves = [c[k].cuda().requires_grad_() for k in ("x", "off", "w", "b")]
    return fn, leaves, (c["stride"], c["pad"], c["dil"], c["cpg"], c["groups"]), c["gout"].cuda()


def _results(fn, leaves, cfg, gout):
    out = fn.apply(*leaves, *cfg)
    return [out] + list(torch.autograd.grad(out, leaves, gout))


def _same(got, want):
    """Equal but for the float atomics that grad_input and grad_offset end in."""
    for g, w in zip(got, want):
        assert g.shape == w.shape and (g - w).norm().item() <= 1e-5 * w.norm().item()


@pytest.mark.parametrize("name", LAYERS)
def test_derived_class_matches_the_function(name):
    print("derived", name, flush=True)
    fn, leaves, cfg, gout = _layer(name)
    derived = type("Derived", (fn,), {})
    assert derived.apply(*leaves, *cfg).grad_fn.name() == "DerivedBackward"
    _same(_results(derived, leaves, cfg, gout), _results(fn, leaves, cfg, gout))


@pytest.mark.parametrize("name", LAYERS)
def test_trace_replays_the_layer(name):
    """A recorded layer gives the layer's results on other inputs, and its gradients."""
    print("trace", name, flush=True)
    fn, leaves, cfg, gout = _layer(name)
    traced = torch.jit.trace(lambda *t: fn.apply(*t, *cfg) * 2, [t.detach() for t in leaves], check_trace=False)
    assert fn.__name__ in str(traced.graph)
    for k in range(2):
        other = [(t.detach() * (1 + k) + 0.25).requires_grad_() for t in leaves]
        out = traced(*other)
        want = fn.apply(*other, *cfg) * 2
        assert torch.equal(out, want)
        _same(torch.autograd.grad(out, other, gout), torch.autograd.grad(want, other, gout))


def test_traced_module():
    import deform_conv3d_pytorch_op_amd as dcn
    print("traced module", flush=True)
    m = torch.nn.Sequential(dcn.ConvOffset2dPack(4, 6, 3, padding=1, channel_per_group=4), torch.nn.ReLU()).cuda()
    x = torch.randn(2, 4, 9, 8, generator=torch.Generator().manual_seed(1)).cuda()
    traced = torch.jit.trace(m, x)
    assert torch.equal(traced(x), m(x)) and torch.equal(traced(x + 1), m(x + 1))


@pytest.mark.parametrize("name", LAYERS)
def test_forward_mode_is_refused(name):
    import torch.autograd.forward_ad as fwad
    print("forward mode", name, flush=True)
    fn, leaves, cfg, _ = _layer(name)
    for at in range(len(leaves)):
        with fwad.dual_level():
            args = [t.detach() for t in leaves]
            args[at] = fwad.make_dual(args[at], torch.ones_like(args[at]))
            with pytest.raises(NotImplementedError, match="jvp"):
                fn.apply(*args, *cfg)
    assert fn.apply(*leaves, *cfg).grad_fn is not None


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, t):
        return t.sum()

    @staticmethod
    def backward(ctx, grad_output):
        return None


@pytest.mark.parametrize("name", LAYERS)
def test_an_undefined_gradient_is_zeros(name):
    """... as it is for a Function: the gradients are there, and zero."""
    print("undefined gradient", name, flush=True)
    fn, leaves, cfg, _ = _layer(name)
    _NoGradient.apply(fn.apply(*leaves, *cfg)).backward()
    for t in leaves:
        assert t.grad is not None and t.grad.shape == t.shape and not t.grad.any()


def test_misshapen_grad_output_is_refused():
    """backward called by hand: no kernel runs on a grad_output that is not the output's shape."""
    import deform_conv3d_pytorch_op_amd as dcn
    from deform_conv3d_pytorch_op_amd import _lib
    for name in LAYERS:
        fn, leaves, cfg, gout = _layer(name)
        leaves = [t.detach() for t in leaves[:-1]]
        for bad, msg in ((gout[:1, :, :-1], "output b|off|outhh|output ll"), (gout[:, :-1], "ou c != ker c"), (gout[..., :-1], "off w|outww"), (gout[0], "output dim")):
            print("misshapen", name, tuple(bad.shape), flush=True)
            with pytest.raises(RuntimeError, match=msg):
                if fn is dcn.Conv2dFunction:
                    _lib.native().conv2d_backward(*leaves, bad, *cfg, True, True, True)
                else:
                    _lib.native().conv_offset_backward(3 if name == "3d" else 2, *leaves, bad, *cfg, False, False, True, True, True)


@pytest.mark.parametrize("name", LAYERS)
def test_saved_tensor_hooks(name):
    """The node saves its tensors through the hooks in force, once each, and gets them back for backward."""
    print("saved-tensor hooks", name, flush=True)
    fn, leaves, cfg, gout = _layer(name)
    want = _results(fn, leaves, cfg, gout)
    packed = []

    def pack(t):
        packed.append(t)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        out = fn.apply(*leaves, *cfg)
    assert {t.data_ptr() for t in packed} == {t.data_ptr() for t in leaves[:-1]} and len(packed) == len(leaves) - 1
    _same([out] + list(torch.autograd.grad(out, leaves, gout)), want)


@pytest.mark.parametrize("reentrant", [False, True])
def test_checkpoint(reentrant):
    import torch.utils.checkpoint as cp
    print("checkpoint", reentrant, flush=True)
    fn, leaves, cfg, gout = _layer("3d")
    out = cp.checkpoint(lambda *t: fn.apply(*t, *cfg).relu(), *leaves, use_reentrant=reentrant)
    want = fn.apply(*leaves, *cfg).relu()
    out.backward(gout)
    _same([t.grad for t in leaves], torch.autograd.grad(want, leaves, gout))


def test_saved_tensor_changed_in_place_is_noticed():
    fn, leaves, cfg, gout = _layer("2d")
    out = fn.apply(*leaves, *cfg)
    with torch.no_grad():
        leaves[2].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(gout)
