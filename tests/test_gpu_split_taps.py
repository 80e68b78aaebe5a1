"""Implicit-GEMM boxes of any extents, and taps of the outermost axes as chunks (the halo in LDS
does not extend along them), against the float64 oracle; the host plan check first. The plan is
asserted, so that each case keeps reaching the path it is here for."""

import ctypes
import math

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, conv_nd, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, dilation, groups, dtype
CASES = {
    # Rank 6: one and two split axes; stride and dilation along them, padding past the taps.
    "rank6_fp32": ((1, 8, 4, 4, 4, 4, 4, 4), (16, 8, 3, 3, 3, 3, 3, 3), (1,) * 6, (1,) * 6, (1,) * 6, 1, torch.float32),
    "rank6_bf16": ((1, 8, 4, 5, 4, 4, 4, 4), (16, 8, 3, 3, 3, 3, 3, 3), (1,) * 6, (1,) * 6, (1,) * 6, 1, torch.bfloat16),
    "rank6_strided": ((1, 8, 5, 6, 3, 4, 3, 4), (8, 8, 3, 2, 3, 2, 3, 3), (2, 1, 1, 2, 1, 1), (1, 0, 1, 1, 1, 1),
                      (1, 2, 1, 1, 1, 1), 1, torch.float32),
    # (The rank-5 one's halo fits LDS in no power-of-two box of 128 positions.)
    "strided_rank5": ((1, 16, 7, 7, 5, 6, 5), (32, 16, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1, torch.bfloat16),
    # Ragged extents: boxes that are no powers of two, idle lanes, partial runs of four.
    "ragged": ((2, 24, 7, 5, 6, 11), (24, 24, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1, torch.bfloat16),
    "ragged_fp32": ((1, 16, 5, 7, 5, 9), (24, 16, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1, torch.float32),
    "one_position": ((1, 16, 3, 3, 3, 3), (16, 16, 3, 3, 3, 3), (1,) * 4, (0,) * 4, (1,) * 4, 1, torch.float16),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


@pytest.mark.parametrize("name", list(CASES))
def test_split_taps_and_boxes(name):
    x_shape, w_shape, stride, padding, dilation, groups, dtype = CASES[name]
    print(f"[taps] {name} {dtype} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    prob = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    assert lib.convnd_hip_plan_check(ctypes.byref(prob), _capi.dtype_code(dtype)) == _capi.SUCCESS
    plans = _capi.plan_details(lib, x_shape, w_shape, stride, padding, dilation, groups, dtype)[:2]
    assert all(p["kernel"] == "mfma_igemm" for p in plans), plans
    if name.startswith("rank"):
        assert any(p["tsplit"] > 0 for p in plans), plans
    if name.startswith("ragged"):
        assert any(math.log2(e) % 1 for p in plans for e in p["box"]), plans
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, dtype, seed=51)
    ref_y = helpers.oracle_forward(x, w, b, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(52)).to(dtype)
    refs = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)
    dev = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = conv_nd(*dev, stride, padding, dilation, groups, backend="native")
    helpers.assert_close(y, ref_y, dtype, f"{name} forward")
    grads = torch.autograd.grad(y, dev, dy.cuda())
    for what, got, want in zip(("grad_input", "grad_weight", "grad_bias"), grads, refs):
        helpers.assert_close(got, want, dtype, f"{name} {what}")
