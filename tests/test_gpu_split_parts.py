"""Split-precision fp32 from the three bf16 parts of each operand (implicit GEMM), layers wider
than 64 channels among them, against the float64 oracle; the host plan check first."""

import ctypes

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, conv_nd, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, dilation, groups
SHAPES = {
    # Channels per part: under, at and over an octet, three octets (one chunk of 24), five.
    "c3": ((1, 3, 4, 5, 6, 7), (17, 3, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "c8_one_tap": ((2, 8, 3, 4, 5, 6), (16, 8, 1, 1, 1, 1), (1,) * 4, (0,) * 4, (1,) * 4, 1),
    "c9": ((1, 9, 4, 3, 5, 6), (8, 9, 2, 3, 2, 3), (1,) * 4, (1,) * 4, (1, 1, 1, 2), 1),
    "c24": ((2, 24, 5, 3, 4, 7), (48, 24, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "c40_groups_strided": ((1, 80, 5, 4, 5, 6), (66, 40, 3, 2, 3, 3), (2, 1, 1, 2), (1, 0, 1, 1), (1,) * 4, 2),
    # Wider than 64 channels in the forward (16 outputs at least), in the input gradient, in both.
    "wide_forward": ((1, 72, 4, 4, 4, 8), (16, 72, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "wide_grad_input": ((1, 17, 4, 3, 4, 5), (100, 17, 2, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "wide_both_strided": ((1, 96, 5, 4, 4, 5), (130, 96, 2, 2, 3, 2), (1, 2, 1, 2), (0, 1, 1, 1), (1,) * 4, 1),
    # Fewer outputs than that: the direct forward.
    "wide_narrow_output": ((1, 72, 3, 3, 4, 5), (15, 72, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


@pytest.mark.parametrize("name", list(SHAPES))
def test_split_parts(name):
    x_shape, w_shape, stride, padding, dilation, groups = SHAPES[name]
    print(f"[split] {name} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    prob = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    assert lib.convnd_hip_plan_check(ctypes.byref(prob), _capi.FLOAT32) == _capi.SUCCESS
    names = _capi.plan_names(lib, x_shape, w_shape, stride, padding, dilation, groups, torch.float32)
    assert names[:2] == ("direct" if name == "wide_narrow_output" else "mfma", "mfma"), names
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.float32, seed=31)
    ref_y = helpers.oracle_forward(x, w, b, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(32))
    refs = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)
    dev = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = conv_nd(*dev, stride, padding, dilation, groups, backend="native")
    helpers.assert_close(y, ref_y, torch.float32, f"{name} forward")
    grads = torch.autograd.grad(y, dev, dy.cuda())
    for what, got, want in zip(("grad_input", "grad_weight", "grad_bias"), grads, refs):
        helpers.assert_close(got, want, torch.float32, f"{name} {what}")


def test_split_parts_infinities():
    """Products with infinities keep the sign of x*w in the three-part layout too."""
    x, w, _ = helpers.seeded_problem((1, 72, 3, 4, 3, 5), (16, 72, 3, 3, 3, 3), False, torch.float32, seed=33)
    x[0, 5, 1, 2, 1, 2] = float("inf")
    x[0, 70, 2, 1, 0, 4] = -float("inf")
    ref = helpers.oracle_forward(x, w, None, (1,) * 4, (1,) * 4, (1,) * 4, 1)
    y = conv_nd(x.cuda(), w.cuda(), None, 1, 1, backend="native").cpu().double()
    ref = torch.as_tensor(ref, dtype=torch.float64)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y), torch.isinf(ref))
    inf = torch.isinf(ref)
    assert torch.equal(y[inf], ref[inf])
