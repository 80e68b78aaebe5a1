"""Performance cases of the N-d convolution: what a program built on this package runs.

A case is one layer call through the public entry points: a training pass (forward, then the
gradients of the input, weight and bias) through ``Conv4d`` / ``ConvNd``, or an inference pass
(``conv_nd`` or the layer without autograd, with or without a fused activation). The listed
cases are the layer shapes of this repository's benchmark and tests plus the calls that a
network made of such layers also holds: its first layer (few input channels), a downsampling
layer, ragged sizes, a large layer and a very small one. ``draw`` spreads over the same ranges.
"""

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "torch-convnd_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import torch_convnd  # noqa: E402

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def _axes(text):
    return tuple(int(v) for v in text.split("x"))


def _case(mode, dtype, batch, cin, cout, size, kernel, stride=None, padding=None, dilation=None,
          groups=1, bias=True, layout="first", activation="none", name=None):
    rank = len(size)
    text = lambda v, default: "x".join(str(a) for a in (v if v is not None else (default,) * rank))  # noqa: E731
    case = {} if name is None else {"name": name}
    case.update(
        mode=mode, dtype=dtype, batch=batch, cin=cin, cout=cout, size=text(size, 0), kernel=text(kernel, 0),
        stride=text(stride, 1), padding=text(padding, 0), dilation=text(dilation, 1), groups=groups, bias=bias,
        layout=layout, activation=activation,
    )
    return case


def listed():
    """``mode``: "train" (forward and every gradient), "train_first" (a network's first layer:
    its input needs no gradient) or "infer" (forward without autograd)."""
    one4, one5, one6 = (1,) * 4, (1,) * 5, (1,) * 6
    return [
        # The smallest training step: a float32 layer of a few channels, bound by launches.
        _case("train", "fp32", 4, 2, 8, (8, 8, 8, 16), (3,) * 4, padding=one4, name="conv4d_fp32_tiny_train"),
        # The smallest inference call: one sample of a small volume, bound by latency.
        _case("infer", "bf16", 1, 16, 16, (6, 6, 6, 6), (3,) * 4, padding=one4, activation="relu",
              name="conv4d_bf16_small_infer"),
        # The ordinary 4-D layer of a bf16 network in training (the benchmark's headline layer).
        _case("train", "bf16", 2, 32, 64, (16,) * 4, (3,) * 4, padding=one4, name="conv4d_bf16_train"),
        # A 5-D layer in training.
        _case("train", "bf16", 1, 16, 32, (12,) * 5, (3,) * 5, padding=one5, name="conv5d_bf16_train"),
        # A 6-D layer in training, in full and in half precision.
        _case("train", "fp32", 1, 8, 16, (8,) * 6, (3,) * 6, padding=one6, name="conv6d_fp32_train"),
        _case("train", "bf16", 1, 8, 16, (8,) * 6, (3,) * 6, padding=one6, name="conv6d_bf16_train"),
        # An anisotropic grouped layer: strided on three axes, dilated on the last.
        _case("train", "bf16", 2, 64, 128, (24, 24, 24, 12), (3, 3, 3, 5), stride=(2, 2, 2, 1),
              padding=(1, 1, 1, 4), dilation=(1, 1, 1, 2), groups=4, bias=False,
              name="conv4d_bf16_grouped_strided_train"),
        # A large layer: many positions and channels, bound by the matrix cores.
        _case("train", "fp16", 4, 64, 64, (24,) * 4, (3,) * 4, padding=one4, name="conv4d_fp16_large_train"),
        # A default-dtype (float32) layer on a ragged volume.
        _case("train", "fp32", 2, 24, 48, (13, 11, 10, 15), (3,) * 4, padding=one4, name="conv4d_fp32_ragged_train"),
        # A network's first layer: three input channels, no input gradient, odd extents.
        _case("train_first", "bf16", 2, 3, 32, (15, 15, 17, 19), (3,) * 4, padding=one4,
              name="conv4d_bf16_first_layer_train"),
        # A downsampling layer: stride 2 on every axis.
        _case("train", "fp16", 2, 32, 64, (20,) * 4, (3,) * 4, stride=(2,) * 4, padding=one4,
              name="conv4d_fp16_downsample_train"),
        # Inference of a layer whose channel counts are no power of two, with a fused activation.
        _case("infer", "bf16", 1, 20, 36, (9, 13, 11, 14), (3,) * 4, padding=one4, activation="gelu",
              name="conv4d_bf16_odd_channels_infer"),
    ]


def _draw_channels(rng):
    c = int(round(math.exp(rng.uniform(math.log(1), math.log(128)))))
    return max(8, c // 8 * 8) if rng.random() < 0.6 else c


def _draw_once(rng):
    rank = rng.choice([4, 4, 4, 4, 5, 5, 6])
    mode = rng.choice(["train", "train", "train", "train_first", "infer", "infer"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32", "fp32"])
    batch = rng.choice([1, 1, 2, 2, 3, 4])
    cin, cout = _draw_channels(rng), _draw_channels(rng)
    groups = 1
    if mode == "train_first":
        cin = rng.randint(1, 4)
    kind = rng.choice(["same", "same", "same", "valid", "pointwise", "strided", "strided", "grouped"])
    k = rng.choice([3, 3, 3, 5]) if rank == 4 else 3
    kernel, stride, padding, dilation = [k] * rank, [1] * rank, [k // 2] * rank, [1] * rank
    if kind == "same" and rng.random() < 0.2:
        dilation[-1] = 2
        padding[-1] = 2 * (k // 2)
    elif kind == "valid":
        kernel = [rng.choice([2, 3]) for _ in range(rank)]
        padding = [0] * rank
    elif kind == "pointwise":
        kernel, padding = [1] * rank, [0] * rank
    elif kind == "strided":
        kernel, padding = [3] * rank, [1] * rank
        stride = [2] * rank if rng.random() < 0.7 else [rng.choice([1, 2]) for _ in range(rank)]
    elif kind == "grouped" and mode != "train_first":
        if rng.random() < 0.4:  # depthwise
            groups = cin = cout = max(4, min(64, cin))
        else:
            groups = rng.choice([2, 4])
            cin, cout = max(1, cin // groups) * groups, max(1, cout // groups) * groups
    # Extents around a common one, odd ones among them, from 4 up to what the rank allows.
    top = {4: 26, 5: 13, 6: 8}[rank]
    base = math.exp(rng.uniform(math.log(4), math.log(top)))
    size = [max(4, min(top, int(round(base * rng.uniform(0.75, 1.3))))) for _ in range(rank)]
    infer = mode == "infer"
    return _case(
        mode, dtype, batch, cin, cout, size, kernel, stride, padding, dilation, groups, rng.random() < 0.8,
        layout="last" if dtype != "fp32" and infer and rng.random() < 0.25 else "first",
        activation=rng.choice(["none", "relu", "gelu"]) if infer else "none",
    )


def draw(rng):
    """One more case of the same ranges: ranks 4 to 6, 1 to 128 channels, extents from 4 up, at
    most about the multiply-adds of the larger listed layers."""
    while True:
        case = _draw_once(rng)
        if 2e5 < _macs(case) < 2.5e10 and work(case)["bytes"] < 1e9:
            return case


def _shapes(case):
    size, kernel = _axes(case["size"]), _axes(case["kernel"])
    stride, padding, dilation = _axes(case["stride"]), _axes(case["padding"]), _axes(case["dilation"])
    out = tuple((n + 2 * p - d * (k - 1) - 1) // s + 1
                for n, k, s, p, d in zip(size, kernel, stride, padding, dilation))
    x_shape = (case["batch"], case["cin"], *size)
    w_shape = (case["cout"], case["cin"] // case["groups"], *kernel)
    return x_shape, w_shape, (case["batch"], case["cout"], *out), stride, padding, dilation


def _macs(case):
    """Multiply-adds of the forward pass whose input sample lies inside the input (padding
    needs none): per axis the (output, tap) pairs with 0 <= o*s - p + t*d < n."""
    x_shape, w_shape, y_shape, stride, padding, dilation = _shapes(case)
    pairs = 1
    for n, k, o, s, p, d in zip(x_shape[2:], w_shape[2:], y_shape[2:], stride, padding, dilation):
        pairs *= sum(1 for i in range(o) for t in range(k) if 0 <= i * s - p + t * d < n)
    return case["batch"] * case["cout"] * w_shape[1] * pairs


def work(case):
    """Each tensor read or written once; two operations per multiply-add inside the input."""
    x_shape, w_shape, y_shape = _shapes(case)[:3]
    nx, nw, ny = math.prod(x_shape), math.prod(w_shape), math.prod(y_shape)
    nb = case["cout"] if case["bias"] else 0
    elements, passes = nx + nw + nb + ny, 1
    if case["mode"] != "infer":
        elements += ny + nw + nb  # grad_output read, weight and bias gradients written
        passes += 1
        if case["mode"] == "train":
            elements += nx
            passes += 1
    return {"bytes": elements * (4 if case["dtype"] == "fp32" else 2), "flops": 2 * passes * _macs(case)}


def _last(t):
    """The same values, stored [N, *spatial, C]."""
    order = (0, *range(2, t.dim()), 1)
    return t.permute(order).contiguous().permute(0, t.dim() - 1, *range(1, t.dim() - 1))


def prepare(case, seed):
    """The layer, its input (unit-variance activations) and, for training, the gradient that
    reaches its output."""
    dtype = _DTYPES[case["dtype"]]
    x_shape, w_shape, y_shape, stride, padding, dilation = _shapes(case)
    torch.manual_seed(seed)
    options = dict(stride=stride, padding=padding, dilation=dilation, groups=case["groups"], bias=case["bias"],
                   device="cuda", dtype=dtype)
    rank = len(x_shape) - 2
    if rank == 4:
        layer = torch_convnd.Conv4d(case["cin"], case["cout"], w_shape[2:], **options)
    else:
        layer = torch_convnd.ConvNd(case["cin"], case["cout"], w_shape[2:], dimensions=rank, **options)
    x = torch.randn(x_shape, device="cuda", dtype=dtype)
    if case["layout"] == "last":
        x = _last(x)
    state = {"case": case, "layer": layer, "x": x}
    if case["mode"] != "infer":
        x.requires_grad_(case["mode"] == "train")
        state["wanted"] = [t for t in (x if case["mode"] == "train" else None, layer.weight, layer.bias)
                           if t is not None]
        state["grad_output"] = torch.randn(y_shape, device="cuda", dtype=dtype)
    return state


def run(state):
    case, layer, x = state["case"], state["layer"], state["x"]
    if case["mode"] == "infer":
        with torch.no_grad():
            if case["activation"] == "none" and case["layout"] == "first":
                return {"y": layer(x)}
            return {"y": torch_convnd.conv_nd(
                x, layer.weight, layer.bias, layer.stride, layer.padding, layer.dilation, layer.groups,
                activation=None if case["activation"] == "none" else case["activation"],
                memory_format=torch.preserve_format if case["layout"] == "last" else torch.contiguous_format,
            )}
    y = layer(x)
    grads = torch.autograd.grad(y, state["wanted"], state["grad_output"])
    names = (("grad_input",) if case["mode"] == "train" else ()) + ("grad_weight", "grad_bias")
    return {"y": y, **dict(zip(names, grads))}


def tolerance(case):
    """16-bit outputs are one rounding of a float32 sum: their error against 64-bit sums is
    1.7e-3 (bf16) and 2.1e-4 (fp16), and one more unit in the last place at most between two
    correct implementations. float32: sums of up to 10^5 products in another order."""
    if case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 4e-2}
    if case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 6e-3}
    return {"rel": 1e-5, "max": 2e-4}


def exact(case, seed):
    """The same outputs in float64: one product per tap of the strided, zero-padded input."""
    state = prepare(case, seed)
    x_shape, w_shape, y_shape, stride, padding, dilation = _shapes(case)
    groups, batch = case["groups"], case["batch"]
    layer, x = state["layer"], state["x"].detach().double()
    train = case["mode"] != "infer"
    pads = [p for a in reversed(padding) for p in (a, a)]
    xp = torch.nn.functional.pad(x, pads)
    w = layer.weight.detach().double().reshape(groups, case["cout"] // groups, w_shape[1], -1)
    y = torch.zeros((batch, groups, case["cout"] // groups, math.prod(y_shape[2:])), dtype=torch.float64,
                    device="cuda")
    if train:
        gy = state["grad_output"].double().reshape(y.shape)
        gw = torch.zeros_like(w)
        gxp = torch.zeros_like(xp) if case["mode"] == "train" else None
    for t in range(w.shape[-1]):
        at, rest = [], t
        for k in reversed(w_shape[2:]):
            at.insert(0, rest % k)
            rest //= k
        window = (slice(None), slice(None)) + tuple(
            slice(a * d, a * d + (o - 1) * s + 1, s) for a, d, o, s in zip(at, dilation, y_shape[2:], stride))
        xt = xp[window].reshape(batch, groups, w_shape[1], -1).contiguous()
        wt = w[..., t].contiguous()
        y += torch.matmul(wt, xt)
        if train:
            gw[..., t] = torch.matmul(gy, xt.transpose(-1, -2).contiguous()).sum(0)
            if gxp is not None:
                gxp[window] += torch.matmul(wt.transpose(-1, -2).contiguous(), gy).reshape(xp[window].shape)
    if case["bias"]:
        y += layer.bias.detach().double().reshape(groups, -1, 1)
    y = y.reshape(y_shape)
    if case["activation"] == "relu":
        y = y.relu()
    elif case["activation"] == "gelu":
        y = torch.nn.functional.gelu(y)
    outputs = {"y": y}
    if case["mode"] == "train":
        inside = (slice(None), slice(None)) + tuple(slice(p, p + n) for p, n in zip(padding, x_shape[2:]))
        outputs["grad_input"] = gxp[inside].contiguous()
    if train:
        outputs["grad_weight"] = gw.reshape(w_shape)
        if case["bias"]:
            outputs["grad_bias"] = gy.sum((0, 3)).reshape(-1)
    return outputs
