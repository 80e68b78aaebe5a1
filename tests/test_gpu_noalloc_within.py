"""The allocation-free forward of a layer whose own plan needs more than its scratch: another plan
runs (marked ``gpu``). Against ``convnd_hip_forward``, which adds in another order."""

import ctypes

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, load_native

pytestmark = pytest.mark.gpu


def test_noalloc_plan_within_its_scratch():
    load_native()
    lib = _build.hip_library()
    x_shape, w_shape, one = (8, 40, 7, 7, 7, 7, 7, 7), (16, 40, 3, 3, 2, 3, 1, 2), (1,) * 6
    problem = _capi.Problem.make(x_shape, w_shape, one, (3, 1, 1, 2, 0, 0), (3, 1, 3, 2, 3, 1), 1)
    ref = ctypes.byref(problem)
    need = lib.convnd_hip_forward_workspace_size(ref, _capi.BFLOAT16)
    assert need > _capi.NOALLOC_SCRATCH_BYTES
    print(f"[noalloc within] x={x_shape} w={w_shape} bf16", flush=True)
    x, w, b = (t.cuda() for t in helpers.seeded_problem(x_shape, w_shape, True, torch.bfloat16, seed=71))
    sizes = (ctypes.c_int64 * _capi.MAX_RANK)()
    assert lib.convnd_hip_validate(ref, 2, 1 << 62, sizes) == _capi.SUCCESS
    want = torch.empty((8, 16, *sizes[:6]), dtype=torch.bfloat16, device="cuda")
    got = torch.full_like(want, float("nan"))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.convnd_hip_forward(ref, _capi.BFLOAT16, ptr(x), ptr(w), ptr(b), ptr(want), ptr(ws), need,
                                  stream) == _capi.SUCCESS
    for _ in range(2):
        got.fill_(float("nan"))
        assert lib.convnd_hip_forward_noalloc(ref, _capi.BFLOAT16, ptr(x), ptr(w), ptr(b), ptr(got),
                                              stream) == _capi.SUCCESS, lib.convnd_hip_last_error().decode()
        helpers.assert_close(got, want.double().cpu(), torch.bfloat16, "noalloc within its scratch")
