"""Forwards of a few products per output (marked ``gpu``): the direct kernel without an activation,
the implicit GEMM with one, against the float64 oracle; channels-last and allocation-free calls
bit for bit as the channels-first one."""

import ctypes

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, conv_nd, load_native

pytestmark = pytest.mark.gpu

CASES = {
    "pointwise": ((1, 1, 4, 3, 5, 2, 3), (72, 1, 1, 1, 1, 1, 1)),
    "two_taps": ((2, 1, 5, 4, 3, 6), (40, 1, 2, 1, 1, 1)),
    "four_channels": ((1, 4, 4, 4, 4, 4), (60, 4, 1, 1, 1, 1)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_few_products(name):
    load_native()
    lib = _build.hip_library()
    x_shape, w_shape = CASES[name]
    rank = len(x_shape) - 2
    args = ((1,) * rank, (0,) * rank, (1,) * rank, 1)
    print(f"[one launch] {name} x={x_shape} w={w_shape}", flush=True)
    assert _capi.plan_names(lib, x_shape, w_shape, *args, torch.bfloat16)[0] == "direct"
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=91)
    ref = helpers.oracle_forward(x, w, b, *args)
    x, w, b = x.cuda(), w.cuda(), b.cuda()
    y = conv_nd(x, w, b, *args, backend="native")
    helpers.assert_close(y, ref, torch.bfloat16, f"{name} forward")
    with torch.no_grad():
        helpers.assert_close(conv_nd(x, w, b, *args, backend="native", activation="gelu"),
                             torch.nn.functional.gelu(ref), torch.bfloat16, f"{name} gelu")
    order = (0, *range(2, rank + 2), 1)
    last = x.permute(order).contiguous().permute(0, rank + 1, *range(1, rank + 1))
    for form in (torch.contiguous_format, torch.preserve_format):
        assert torch.equal(conv_nd(last, w, b, *args, backend="native", memory_format=form), y)
    got = torch.full_like(y, float("nan"))
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    problem = _capi.Problem.make(x_shape, w_shape, *args)
    assert lib.convnd_hip_forward_noalloc(ctypes.byref(problem), _capi.BFLOAT16, ptr(x), ptr(w), ptr(b), ptr(got),
                                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert torch.equal(got, y)
