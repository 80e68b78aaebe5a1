"""Split-precision fp32 staging: the three parts of every run from one read of the source
(octet-major copies, zero-padded copies of grad_output and of the input), against the float64
oracle at the edges of its runs and blocks."""

import pytest
import torch

import helpers
from torch_convnd import conv_nd, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, groups
SHAPES = {
    # 1023, 1024 and 1025 positions: a block of the octet copy is 1024.
    "volume_1023": ((1, 9, 3, 11, 31), (24, 9, 3, 3, 3), (1,) * 3, (1,) * 3, 1),
    "volume_1024": ((2, 16, 4, 16, 16), (16, 16, 3, 3, 3), (1,) * 3, (1,) * 3, 1),
    "volume_1025": ((1, 8, 5, 5, 41), (17, 8, 3, 3, 3), (1,) * 3, (1,) * 3, 1),
    # Channels that end inside an octet, in each of three groups, three images.
    "groups": ((3, 33, 4, 5, 3, 6), (42, 11, 3, 3, 2, 3), (1,) * 4, (1, 1, 0, 1), 3),
    # One image row shorter than a run, and an even kernel on the last axis (one copy shift).
    "short_rows": ((2, 12, 6, 5, 4, 3), (20, 12, 3, 3, 3, 2), (1,) * 4, (1, 1, 1, 0), 1),
    # Strided: the input gradient's phases and, on the last axis, the copies per phase.
    "strided": ((2, 24, 6, 5, 7, 9), (40, 24, 3, 3, 3, 3), (1, 2, 1, 2), (1,) * 4, 1),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_split_prologue(name):
    load_native()
    x_shape, w_shape, stride, padding, groups = SHAPES[name]
    print(f"[split prologue] {name} x={x_shape} w={w_shape}", flush=True)
    dilation = (1,) * len(stride)
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.float32, seed=71)
    ref_y = helpers.oracle_forward(x, w, b, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(72))
    refs = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)
    dev = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = conv_nd(*dev, stride, padding, dilation, groups, backend="native")
    helpers.assert_close(y, ref_y, torch.float32, f"{name} forward")
    grads = torch.autograd.grad(y, dev, dy.cuda())
    for what, got, want in zip(("grad_input", "grad_weight", "grad_bias"), grads, refs):
        helpers.assert_close(got, want, torch.float32, f"{name} {what}")
