"""Layers whose channel counts are no whole octets on the implicit GEMM (16-bit data): the
staged GEMM input holds zero channels up to the next octet. Forward and every gradient against
the float64 oracle, with the host plan check first; the call forms without scratch or tables."""

import ctypes

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, conv_nd, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, dilation, groups
SHAPES = {
    "one_over_an_octet": ((1, 9, 3, 4, 5, 6), (16, 9, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "one_under_an_octet": ((2, 15, 4, 3, 4, 9), (33, 15, 2, 3, 2, 3), (1,) * 4, (0, 1, 1, 2), (1,) * 4, 1),
    "first_layer": ((2, 3, 5, 5, 7, 9), (32, 3, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "single_channel": ((1, 1, 5, 6, 4, 7), (40, 1, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "head": ((1, 32, 4, 5, 4, 7), (3, 32, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    "groups": ((2, 20, 4, 4, 5, 6), (36, 5, 3, 2, 3, 3), (1,) * 4, (1,) * 4, (1, 1, 1, 2), 4),
    "strided": ((2, 6, 7, 5, 6, 9), (10, 6, 3, 3, 3, 3), (2, 1, 2, 2), (1,) * 4, (1,) * 4, 1),
    "rank5": ((1, 12, 3, 4, 3, 4, 5), (20, 12, 3, 3, 2, 3, 3), (1,) * 5, (1, 1, 0, 1, 1), (1,) * 5, 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("name", list(SHAPES))
def test_padded_channels(name, dtype):
    x_shape, w_shape, stride, padding, dilation, groups = SHAPES[name]
    print(f"[padded] {name} {dtype} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    prob = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    assert lib.convnd_hip_plan_check(ctypes.byref(prob), _capi.dtype_code(dtype)) == _capi.SUCCESS
    names = _capi.plan_names(lib, x_shape, w_shape, stride, padding, dilation, groups, dtype)
    assert names[0] == "mfma" and names[1] == "mfma", names
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, dtype, seed=21)
    ref_y = helpers.oracle_forward(x, w, b, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(22)).to(dtype)
    refs = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)
    dev = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = conv_nd(*dev, stride, padding, dilation, groups, backend="native")
    helpers.assert_close(y, ref_y, dtype, f"{name} forward")
    grads = torch.autograd.grad(y, dev, dy.cuda())
    for what, got, want in zip(("grad_input", "grad_weight", "grad_bias"), grads, refs):
        helpers.assert_close(got, want, dtype, f"{name} {what}")
    # The bias gradient beside the input gradient alone (its own channel sums).
    gx, gb = torch.autograd.grad(conv_nd(*dev, stride, padding, dilation, groups, backend="native"),
                                 (dev[0], dev[2]), dy.cuda())
    assert torch.equal(gx, grads[0])
    helpers.assert_close(gb, refs[2], dtype, f"{name} grad_bias beside grad_input")


def test_padded_channels_last():
    x_shape, w_shape, stride, padding, dilation, groups = SHAPES["groups"]
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=23)
    args = (stride, padding, dilation, groups)
    leaves = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = conv_nd(*leaves, *args, backend="native")
    dy = torch.randn(y.shape, generator=torch.Generator().manual_seed(24)).to(y.dtype).cuda()
    want = torch.autograd.grad(y, leaves, dy)
    last = lambda t: t.permute(0, 2, 3, 4, 5, 1).contiguous().permute(0, 5, 1, 2, 3, 4)  # noqa: E731
    lx = last(x.cuda()).requires_grad_()
    ly = conv_nd(lx, *leaves[1:], *args, backend="native", memory_format=torch.preserve_format)
    got = torch.autograd.grad(ly, (lx, *leaves[1:]), last(dy))
    assert torch.equal(ly, y)
    for a, c in zip(got, want):
        assert torch.equal(a, c)


def test_padded_first_call_under_capture():
    """A geometry never called before stays capturable (the direct kernels need no tables)."""
    x_shape, w_shape = (1, 5, 3, 4, 5, 11), (18, 5, 3, 3, 3, 3)
    one = (1,) * 4
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=25)
    ref = helpers.oracle_forward(x, w, b, one, one, one, 1)
    x, w, b = (t.cuda() for t in (x, w, b))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = torch.ops.torch_convnd.conv_nd(x, w, b, one, one, one, 1, 64 << 20)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        helpers.assert_close(y, ref, torch.bfloat16, "captured first call")


def test_padded_noalloc_beyond_its_scratch():
    """The allocation-free entry point still takes a problem whose staging exceeds its scratch."""
    lib = _build.hip_library()
    x_shape, w_shape = (1, 1, 20, 20, 100, 120), (48, 1, 1, 1, 1, 1)
    one, zero = (1,) * 4, (0,) * 4
    prob = _capi.Problem.make(x_shape, w_shape, one, zero, one, 1)
    assert lib.convnd_hip_forward_workspace_size(ctypes.byref(prob), _capi.BFLOAT16) > _capi.NOALLOC_SCRATCH_BYTES
    x, w, b = (t.cuda() for t in helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=26))
    y = torch.full((1, 48, *x_shape[2:]), float("nan"), dtype=torch.bfloat16, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = lib.convnd_hip_forward_noalloc(ctypes.byref(prob), _capi.BFLOAT16, ptr(x), ptr(w), ptr(b), ptr(y),
                                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == _capi.SUCCESS, lib.convnd_hip_last_error().decode()
    torch.cuda.synchronize()
    want = x.float() * w.float().reshape(1, 48, 1, 1, 1, 1) + b.float().reshape(1, 48, 1, 1, 1, 1)
    helpers.assert_close(y, want.double().cpu(), torch.bfloat16, "noalloc beyond scratch")
