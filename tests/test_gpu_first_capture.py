"""The first call of a geometry under stream capture (marked ``gpu``): its geometry tables cannot be
uploaded then, and layers whose plans may do without run on the direct kernels. Every layout of
the input and output, each replay against the float64 oracle."""

import pytest
import torch

import helpers
from torch_convnd import conv_nd, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, dilation, groups: no power-of-two box of 128 output positions
# holds (the first) or fits LDS with its halo (the others).
CASES = {
    "few_positions": ((1, 32, 2, 3, 2, 4), (32, 32, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "large_halo": ((1, 8, 4, 8, 3, 7, 7, 4), (8, 8, 3, 5, 2, 4, 3, 3), (3, 1, 3, 2, 1, 1), (1, 2, 1, 2, 1, 1),
                   (1,) * 6, 1),
    # (Its bare halo fits, not with its tables.)
    "strided_rank5": ((1, 8, 9, 9, 9, 9, 9), (16, 8, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


def channels_last(t):
    order = (0, *range(2, t.dim()), 1)
    return t.permute(order).contiguous().permute(0, t.dim() - 1, *range(1, t.dim() - 1))


@pytest.mark.parametrize("layout", ["first", "last_input", "last"])
@pytest.mark.parametrize("name", list(CASES))
def test_first_call_under_capture(name, layout):
    x_shape, w_shape, *args = CASES[name]
    # (A batch of its own per layout: each one is the geometry's first call.)
    x_shape = (x_shape[0] + ["first", "last_input", "last"].index(layout), *x_shape[1:])
    print(f"[first capture] {name} {layout} x={x_shape} w={w_shape}", flush=True)
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=61)
    ref = helpers.oracle_forward(x, w, b, *args)
    x, w, b = x.cuda(), w.cuda(), b.cuda()
    if layout != "first":
        x = channels_last(x)
    other = torch.zeros((5, *x_shape[1:]), dtype=x.dtype, device="cuda")
    form = torch.preserve_format if layout == "last" else torch.contiguous_format
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = conv_nd(x, w, b, *args, backend="native", memory_format=form)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        helpers.assert_close(y, ref, torch.bfloat16, f"{name} {layout}: captured first call")
        conv_nd(other, w, b, *args, backend="native")  # another geometry, between the replays
    assert layout != "last" or y.permute(0, *range(2, y.dim()), 1).is_contiguous()


# The gradients that may do without tables: of the input (few positions), of the weight (strided).
@pytest.mark.parametrize(("name", "mask"), [("few_positions", (True, False, True)),
                                            ("strided_rank5", (False, True, True))])
@pytest.mark.parametrize("layout", ["first", "last_input", "last"])
def test_first_backward_under_capture(name, mask, layout):
    x_shape, w_shape, *args = CASES[name]
    x_shape = (x_shape[0] + 6 + ["first", "last_input", "last"].index(layout), *x_shape[1:])
    print(f"[first capture] backward {name} {layout} x={x_shape} w={w_shape}", flush=True)
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=62)
    y = helpers.oracle_forward(x, w, b, *args)
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(63)).to(torch.bfloat16)
    refs = helpers.oracle_backward(dy, x, w, *args)
    x, w, dy = x.cuda(), w.cuda(), dy.cuda()
    if layout != "first":
        x = channels_last(x)
    if layout == "last":
        dy = channels_last(dy)
    ops = torch.ops.torch_convnd
    backward = ops.conv_nd_backward_preserve if layout == "last" else ops.conv_nd_backward
    params = (*map(list, args[:3]), args[3], 1 << 26, list(mask))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        grads = backward(dy, x, w, *params)
    for _ in range(3):
        for g, wanted in zip(grads, mask):
            if wanted:
                g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for what, got, want, wanted in zip(("grad_input", "grad_weight", "grad_bias"), grads, refs, mask):
            if wanted:
                helpers.assert_close(got, want, torch.bfloat16, f"{name} {layout} {what}: captured first call")
        conv_nd(torch.zeros((5, *x_shape[1:]), dtype=x.dtype, device="cuda"), w, None, *args, backend="native")
