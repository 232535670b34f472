"""What a user of this package has it do, as cases that can be timed and compared.

A case is one layer of the package (a module of `deform_conv3d_pytorch_op_amd`) on synthetic inputs:
`mode` "train" is a forward and a backward pass through autograd with every gradient the layer
gives (input, offset, weight, bias), "infer" a forward pass without autograd.  The module, its
parameters and the tensors are what a user's program holds before the call.

Keys: op "deform" (ConvOffset2d / ConvOffset3d) or "conv2d" (the plain Conv2d), nd, dtype, mode,
n, cin, cout, in_l / in_h / in_w (in_l is 1 in 2-D), k, stride_l / stride (along l / along h and w),
pad, dil, cpg (channels per deformable group), groups, offsets ("uniform": U[-reach, reach];
"mix": N(0, 1) with one value in ten from U[-6, 6]), reach, bias.
"""
import math

import torch

import deform_conv3d_pytorch_op_amd as dcn

DTYPES = {"float64": torch.float64, "float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
DEVICE = "cuda:0"


def _case(name=None, op="deform", nd=3, dtype="float32", mode="train", n=1, cin=64, cout=64, size=(16, 56, 56), k=3,
          stride=1, stride_l=1, pad=1, dil=1, cpg=None, groups=1, offsets="uniform", reach=1.5, bias=True):
    size = (1,) * (3 - len(size)) + tuple(size)
    c = dict(op=op, nd=nd, dtype=dtype, mode=mode, n=n, cin=cin, cout=cout, in_l=size[0], in_h=size[1], in_w=size[2], k=k,
             stride=stride, stride_l=stride_l, pad=pad, dil=dil, cpg=cpg or cin, groups=groups, offsets=offsets,
             reach=float(reach), bias=bias)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: the double-precision layer that a gradient check runs over and over
        # (2 images of 16 x 16, 8 -> 8 channels); launches and host work are all of it
        _case("2d f64 gradient check", nd=2, dtype="float64", n=2, cin=8, cout=8, size=(16, 16)),
        # one short clip through a late layer of a video network, one at a time: latency
        _case("3d f32 small clip infer", mode="infer", n=1, cin=32, cout=32, size=(8, 14, 14)),
        # one image of odd size through an early detection layer, one at a time
        _case("2d f32 odd image infer", nd=2, mode="infer", n=1, cin=64, cout=64, size=(75, 101), reach=2.0),
        # training steps of 2-D layers: a wide one in one deformable group, and a dilated one with
        # two convolution groups, four deformable groups and some far-reaching offsets
        _case("2d f32 256ch train", nd=2, n=8, cin=256, cout=256, size=(56, 56), reach=2.0),
        _case("2d f32 512ch groups train", nd=2, n=4, cin=512, cout=512, size=(28, 28), pad=2, dil=2, cpg=128, groups=2,
              offsets="mix"),
        # the package's headline layer: 3-D, 64 channels, a batch of four clips of 16 x 56 x 56
        _case("3d f32 64ch train", n=4),
        _case("3d f32 64ch infer", n=4, mode="infer"),
        # the largest: a strided 3-D layer of 128 channels in four deformable groups
        _case("3d f32 128ch strided train", n=2, cin=128, cout=128, size=(16, 112, 112), stride=2, cpg=32, reach=2.0),
        # nothing divides evenly: odd extents, 48 -> 80 channels in two deformable groups
        _case("3d f32 ragged train", n=2, cin=48, cout=80, size=(11, 37, 29), cpg=24, reach=2.0),
        # training in 16-bit storage
        _case("3d bf16 64ch train", n=4, dtype="bfloat16"),
        _case("2d f16 256ch train", nd=2, n=8, cin=256, cout=256, size=(56, 56), reach=2.0, dtype="float16"),
        # the plain convolution of the package
        _case("conv2d f32 64ch train", op="conv2d", nd=2, n=8, cin=64, cout=64, size=(56, 56)),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """A layer of the same ranges: 2-D and 3-D, every storage type, training and inference, 8 to 512
    (2-D) or 8 to 128 (3-D) channels, from a few hundred positions to tens of thousands, with the kernels, strides,
    dilations and group counts that the listed layers and the tests use.  Its number of samples
    (batch x channels x taps x positions) is drawn over a factor of several hundred and stays well below
    that of the largest listed layer."""
    while True:
        op = "conv2d" if rng.random() < 0.08 else "deform"
        nd = 2 if op == "conv2d" or rng.random() < 0.5 else 3
        dtype = rng.choice(["float32"] * 6 + ([] if op == "conv2d" else ["bfloat16", "bfloat16", "float16"]) + ["float64"])
        groups = rng.choice([1, 1, 1, 1, 2])
        dgroups = 1 if op == "conv2d" else rng.choice([1, 1, 1, 2, 4])
        top = 512 if nd == 2 else 128
        unit = groups * dgroups
        cin = _log_int(rng, 8, top) // unit * unit
        cout = _log_int(rng, 8, top) // groups * groups
        if rng.random() < 0.5:      # half of the layers have the usual multiples of 16
            cin, cout = cin // (16 * unit) * 16 * unit, cout // (16 * groups) * 16 * groups
        if cin < 8 or cout < 8:
            continue
        k = rng.choice([3, 3, 3, 3, 1] if nd == 3 else [3, 3, 3, 3, 1, 5])
        stride = rng.choice([1, 1, 1, 2])
        stride_l = rng.choice([1, stride])
        dil = rng.choice([1, 1, 1, 2]) if k == 3 else 1
        pad = k // 2 * dil
        n = rng.choice([1, 1, 2, 3, 4, 8])
        samples = math.exp(rng.uniform(math.log(3e5), math.log(2.5e7 if dtype == "float64" else 9e7)))
        positions = samples / (n * cin * k ** nd)
        side = positions ** (1 / nd)
        if side < 5 or side > (160 if nd == 2 else 64):
            continue
        flat = math.exp(rng.uniform(-0.3, 0.3)), math.exp(rng.uniform(-0.3, 0.3))
        h = max(5, round(side * flat[0])) * stride
        w = max(5, round(side / flat[0] * flat[1])) * stride
        l = max(3, round(side / flat[1])) * stride_l if nd == 3 else 1
        c = _case(op=op, nd=nd, dtype=dtype, mode=rng.choice(["train", "train", "infer"]), n=n, cin=cin, cout=cout,
                  size=(l, h, w), k=k, stride=stride, stride_l=stride_l, pad=pad, dil=dil, cpg=cin // dgroups, groups=groups,
                  offsets="mix" if rng.random() < 0.1 else "uniform", reach=rng.choice([0.5, 1.0, 1.5, 2.0, 3.0]),
                  bias=rng.random() < 0.75)
        flops = work(c)["flops"]
        if min(_out(c)[3 - nd:]) < 3 or flops > (8e9 if dtype == "float64" else 1.2e11):
            continue
        return c


def _strides(c):
    return (c["stride_l"], c["stride"], c["stride"])[3 - c["nd"]:]


def _out(c):
    """Output extents (l, h, w).  The deformable layers do not count dilation (their own rule), the plain convolution does."""
    span = c["dil"] * (c["k"] - 1) + 1 if c["op"] == "conv2d" else c["k"]
    size = lambda i, s: (i + 2 * c["pad"] - span) // s + 1
    return (size(c["in_l"], c["stride_l"]) if c["nd"] == 3 else 1, size(c["in_h"], c["stride"]), size(c["in_w"], c["stride"]))


def _elems(c):
    kv, out_v = c["k"] ** c["nd"], math.prod(_out(c))
    off = 0 if c["op"] == "conv2d" else c["n"] * (c["cin"] // c["cpg"]) * c["nd"] * kv * out_v
    return dict(x=c["n"] * c["cin"] * c["in_l"] * c["in_h"] * c["in_w"], off=off,
                w=c["cout"] * (c["cin"] // c["groups"]) * kv, b=c["cout"] if c["bias"] else 0, out=c["n"] * c["cout"] * out_v)


def prepare(case, seed):
    c = case
    nd, dtype = c["nd"], DTYPES[c["dtype"]]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    draw_dtype = torch.float64 if dtype == torch.float64 else torch.float32

    def normal(*shape):
        return torch.randn(shape, generator=g, device=DEVICE, dtype=draw_dtype)

    def uniform(reach, *shape):
        return (torch.rand(shape, generator=g, device=DEVICE, dtype=draw_dtype) * 2 - 1) * reach

    kw = dict(stride=_strides(c), padding=c["pad"], dilation=c["dil"], bias=c["bias"], groups=c["groups"], device=DEVICE, dtype=dtype)
    if c["op"] == "conv2d":
        layer = dcn.Conv2d(c["cin"], c["cout"], c["k"], **kw)
    else:
        layer = (dcn.ConvOffset3d if nd == 3 else dcn.ConvOffset2d)(c["cin"], c["cout"], c["k"], channel_per_group=c["cpg"], **kw)
    with torch.no_grad():           # Kaiming-normal (fan out) weights and a small bias, from the seed
        layer.weight.copy_(normal(*layer.weight.shape) * math.sqrt(2.0 / (c["cout"] * c["k"] ** nd)))
        if c["bias"]:
            layer.bias.copy_(uniform(0.1, c["cout"]))
    ins = (c["in_l"], c["in_h"], c["in_w"])[3 - nd:]
    outs = _out(c)[3 - nd:]
    state = dict(layer=layer, train=c["mode"] == "train", deform=c["op"] == "deform")
    x = normal(c["n"], c["cin"], *ins).to(dtype)
    off = None
    if state["deform"]:
        shape = (c["n"], c["cin"] // c["cpg"] * nd * c["k"] ** nd) + outs
        if c["offsets"] == "mix":
            far = torch.rand(shape, generator=g, device=DEVICE, dtype=draw_dtype) < 0.1
            off = torch.where(far, uniform(6.0, *shape), normal(*shape)).to(dtype)
        else:
            off = uniform(c["reach"], *shape).to(dtype)
    if state["train"]:
        state["grad_output"] = normal(c["n"], c["cout"], *outs).to(dtype)
        x.requires_grad_(True)
        if off is not None:
            off.requires_grad_(True)
    state["x"], state["off"] = x, off
    return state


def run(state):
    layer, x, off = state["layer"], state["x"], state["off"]
    args = (x, off) if state["deform"] else (x,)
    if not state["train"]:
        with torch.no_grad():
            return layer(*args)
    x.grad = layer.weight.grad = None
    if off is not None:
        off.grad = None
    if layer.bias is not None:
        layer.bias.grad = None
    out = layer(*args)
    out.backward(state["grad_output"])
    got = dict(output=out.detach(), grad_input=x.grad, grad_weight=layer.weight.grad)
    if off is not None:
        got["grad_offset"] = off.grad
    if layer.bias is not None:
        got["grad_bias"] = layer.bias.grad
    return got


def work(case):
    """The tensors read once and the results written once; the multiply-adds of the dense contractions
    (one in the forward pass, three in a training step)."""
    c, e = case, _elems(case)
    size = DTYPES[c["dtype"]].itemsize
    contraction = 2.0 * c["n"] * c["cout"] * (c["cin"] // c["groups"]) * c["k"] ** c["nd"] * math.prod(_out(c))
    moved = e["x"] + e["off"] + e["w"] + e["b"] + e["out"]
    if c["mode"] == "train":
        moved += e["out"] + e["x"] + e["off"] + e["w"] + e["b"]         # grad_output in, the gradients out
    return {"bytes": float(moved * size), "flops": contraction * (3 if c["mode"] == "train" else 1)}


def tolerance(case):
    """Relative 2-norm.  float32: grad_input is summed in 32-bit fixed point and is 5e-5 away from
    the double-precision result on the 3-D layers (the other results 2e-6), and the rounding depends
    on how positions are grouped.  16-bit storage: one rounding of the sampled values and one of each result."""
    return {"rel": {"float64": 1e-12, "float32": 1e-4, "bfloat16": 1e-2, "float16": 2e-3}[case["dtype"]]}
