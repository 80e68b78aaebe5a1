"""Input gradients of strided convolutions whose stride phases share one staged halo, against the
float64 oracle; the host plan check first. The number of phases per workgroup is forced (the
planner's override is read once per process)."""

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
    # Odd and even extents: phases with fewer positions than the first, boxes past some of them.
    "stride2": ((2, 16, 5, 6, 7, 9), (24, 16, 3, 3, 3, 3), (2,) * 4, (1,) * 4, (1,) * 4, 1),
    # Phases without any tap (stride above the kernel), and with different shifts (even kernel).
    "stride_above_kernel": ((1, 8, 7, 5, 9, 11), (16, 8, 2, 2, 2, 2), (1, 2, 3, 4), (0, 1, 1, 1), (1,) * 4, 1),
    "even_kernel": ((1, 8, 6, 6, 5, 8), (8, 8, 4, 2, 3, 4), (2, 1, 2, 2), (2, 0, 1, 1), (1,) * 4, 1),
    "dilated": ((1, 16, 6, 5, 9, 7), (16, 16, 2, 3, 3, 2), (2, 1, 2, 2), (1, 1, 2, 1), (1, 1, 2, 3), 1),
    "groups": ((2, 16, 6, 5, 6, 10), (48, 8, 3, 3, 3, 3), (2, 2, 1, 2), (1,) * 4, (1,) * 4, 2),
    "rank5": ((1, 16, 5, 4, 6, 5, 7), (32, 16, 3, 3, 3, 3, 3), (2, 2, 1, 2, 2), (1,) * 5, (1,) * 5, 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


def check(name, dtype):
    x_shape, w_shape, stride, padding, dilation, groups = SHAPES[name]
    print(f"[phases] {name} {dtype} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    prob = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    assert lib.convnd_hip_plan_check(ctypes.byref(prob), _capi.dtype_code(dtype)) == _capi.SUCCESS, \
        lib.convnd_hip_last_error()
    plan = _capi.plan_details(lib, x_shape, w_shape, stride, padding, dilation, groups, dtype)[1]
    x, w, b = helpers.seeded_problem(x_shape, w_shape, False, dtype, seed=71)
    ref_y = helpers.oracle_forward(x, w, None, stride, padding, dilation, groups)
    dy = torch.randn(ref_y.shape, generator=torch.Generator().manual_seed(72)).to(dtype)
    ref = helpers.oracle_backward(dy, x, w, stride, padding, dilation, groups)[0]
    gx = torch.ops.torch_convnd.conv_nd_backward(dy.cuda(), x.cuda(), w.cuda(), stride, padding, dilation, groups,
                                                 64 << 20, [True, False, False])[0]
    helpers.assert_close(gx, ref, dtype, f"{name} grad_input")
    return plan["plen"]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("name", list(SHAPES))
def test_planned(name, dtype):
    check(name, dtype)


@pytest.mark.parametrize("plen", [1, 2, 4, 16])
def test_forced_phase_groups(plen):
    code = (
        "import sys; sys.path[:0] = ['tests', 'torch-convnd_amd']\n"
        "import torch, test_gpu_phase_groups as t\n"
        "t.load_native()\n"
        "seen = [t.check(n, d) for n in t.SHAPES for d in (torch.bfloat16, torch.float32)]\n"
        f"assert {plen} in seen, seen\n"
    )
    env = dict(os.environ, CONVND_HIP_DGRAD_PLAN=f"plen={plen}")
    out = subprocess.run([sys.executable, "-u", "-c", code], cwd=Path(__file__).resolve().parent.parent, env=env,
                         capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-2000:]
