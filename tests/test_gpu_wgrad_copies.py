"""Channel-major weight gradient on several copies of the padded input: strided last axes (a copy
per phase) and copies shifted by one element (odd last-axis taps), against the float64 oracle; the
host plan check first."""

import ctypes
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, load_native

pytestmark = pytest.mark.gpu

# x shape, w shape, stride, padding, dilation, groups
SHAPES = {
    "stride2": ((2, 16, 7, 6, 9, 13), (24, 16, 3, 3, 3, 3), (2,) * 4, (1,) * 4, (1,) * 4, 1),
    "stride2_even_kernel": ((1, 8, 6, 5, 6, 18), (16, 8, 2, 2, 2, 4), (2, 1, 2, 2), (0, 1, 0, 3), (1,) * 4, 1),
    "stride3_dilated": ((1, 8, 5, 4, 7, 30), (16, 8, 2, 2, 3, 3), (1, 1, 2, 3), (1, 0, 1, 4), (1, 1, 1, 4), 1),
    "stride4": ((1, 12, 4, 5, 5, 41), (20, 12, 3, 2, 2, 5), (1, 2, 1, 4), (1, 1, 0, 2), (1,) * 4, 1),
    # Beyond the kernel's strides: the octet-major kernel.
    "stride5": ((1, 8, 4, 4, 5, 47), (16, 8, 2, 2, 2, 3), (1, 1, 1, 5), (0,) * 4, (1,) * 4, 1),
    "rank5_stride2": ((1, 16, 7, 7, 5, 6, 9), (32, 16, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1),
    "groups": ((1, 16, 5, 6, 5, 11), (24, 8, 3, 3, 3, 3), (1, 2, 1, 2), (1,) * 4, (1,) * 4, 2),
    "odd_taps": ((1, 8, 4, 4, 4, 4, 5, 9), (16, 8, 3, 3, 3, 3, 3, 3), (1,) * 6, (1,) * 6, (1,) * 6, 1),
    "odd_dilation": ((2, 16, 5, 6, 7, 21), (16, 16, 3, 3, 3, 5), (1,) * 4, (1, 1, 1, 6), (1, 1, 1, 3), 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


def _check(name, dtype):
    x_shape, w_shape, stride, padding, dilation, groups = SHAPES[name]
    print(f"[copies] {name} {dtype} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    prob = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    assert lib.convnd_hip_plan_check(ctypes.byref(prob), _capi.dtype_code(dtype)) == _capi.SUCCESS, \
        lib.convnd_hip_last_error()
    plan = _capi.plan_details(lib, x_shape, w_shape, stride, padding, dilation, groups, dtype)[2]
    if stride[-1] == 1 or name == "rank5_stride2" or "cm=1" in os.environ.get("CONVND_HIP_WGRAD_PLAN", ""):
        assert plan["kernel"] == ("mfma_wgrad" if name == "stride5" else "mfma_wgrad_cm"), plan
    x, w, b = helpers.seeded_problem(x_shape, w_shape, True, dtype, seed=61)
    ref_y = helpers.oracle_forward(x, w, b, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(62)).to(dtype)
    refs = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)
    # An input at a 2-byte-aligned address: the copies take any alignment of the source.
    xd = torch.empty(x.numel() + 8, dtype=dtype, device="cuda")[1 : 1 + x.numel()].view(x_shape).copy_(x)
    for inp in (x.cuda(), xd):
        _, gw, gb = torch.ops.torch_convnd.conv_nd_backward(
            dy.cuda(), inp, w.cuda(), stride, padding, dilation, groups, 64 << 20, [False, True, True])
        helpers.assert_close(gw, refs[1], dtype, f"{name} grad_weight")
        helpers.assert_close(gb, refs[2], dtype, f"{name} grad_bias")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("name", list(SHAPES))
def test_copies(name, dtype):
    _check(name, dtype)


@pytest.mark.parametrize("override", ["parity=0", "parity=1", "cm=1,parity=0", "cm=1,parity=1"])
def test_each_layout(override):
    """Every case on the channel-major kernel, with and without shifted copies, whichever the
    planner prefers (its override is read once per process)."""
    names = list(SHAPES) if "cm" in override else [n for n in SHAPES if SHAPES[n][2][-1] == 1]
    code = (
        "import sys; sys.path[:0] = ['tests', 'torch-convnd_amd']\n"
        "import torch, test_gpu_wgrad_copies as t\n"
        "t.load_native()\n"
        f"for name in {names!r}:\n"
        "    for dtype in (torch.bfloat16, torch.float32):\n"
        "        t._check(name, dtype)\n"
    )
    env = dict(os.environ, CONVND_HIP_WGRAD_PLAN=override)
    out = subprocess.run([sys.executable, "-u", "-c", code], cwd=Path(__file__).resolve().parent.parent, env=env,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-2000:]
