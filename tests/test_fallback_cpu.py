"""Calls whose plan cannot have its geometry tables (without a GPU: every call), on the host.

Without a device the tables of a plan cannot be uploaded, as they cannot on the first call of a
geometry under stream capture: a plan that may run on the direct kernels instead goes on to
them, and its call then fails at the first launch, which the message names. Nothing runs, so the
buffers are addresses that are never read. Skipped where a GPU is present.
"""

import ctypes
import math
import random
import time

import pytest
import torch

from torch_convnd import _capi
from torch_convnd._toolchain import HIP_LIBRARY

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="the calls would run on the GPU")

NOWHERE = ctypes.c_void_p(0x10000)


@pytest.fixture(scope="module")
def lib():
    if not HIP_LIBRARY.exists():
        pytest.skip("native libraries not built (python __graft_entry__.py)")
    return _capi.bind(ctypes.CDLL(str(HIP_LIBRARY)))


def out_shape(lib, problem, x_shape, w_shape):
    sizes = (ctypes.c_int64 * _capi.MAX_RANK)()
    assert lib.convnd_hip_validate(ctypes.byref(problem), 2, 1 << 62, sizes) == _capi.SUCCESS
    return (x_shape[0], w_shape[0], *sizes[: len(x_shape) - 2])


def small_problems(count, seed):
    """16-bit layers of few output positions, or of halos near the size of LDS."""
    rng = random.Random(seed)
    for _ in range(count):
        rank = rng.randint(1, 6)
        top = {1: 60, 2: 20, 3: 16, 4: 11, 5: 11, 6: 6}[rank]
        kernel = [rng.randint(2, 4 if rank < 5 else 3) for _ in range(rank)]
        stride = [rng.choice((1, 1, 2, 3))] * rank
        size = [max(k, rng.randint(2, top)) for k in kernel]
        cin, cout = rng.choice((8, 16, 32, 5)), rng.choice((8, 16, 64, 3))
        yield (rng.choice((1, 2)), cin, *size), (cout, cin, *kernel), tuple(stride), (1,) * rank, (1,) * rank, 1


CHANNELS_LAST_CASES = [
    # Fewer output positions than a tile, and a halo that no box of 128 positions fits.
    ((1, 32, 2, 3, 2, 4), (32, 32, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1),
    ((1, 8, 4, 8, 3, 7, 7, 4), (8, 8, 3, 5, 2, 4, 3, 3), (3, 1, 3, 2, 1, 1), (1, 2, 1, 2, 1, 1), (1,) * 6, 1),
    ((1, 16, 13, 10, 11, 11, 8), (8, 16, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1),
    *small_problems(150, 3),
]


def test_channels_last_forward_stays_inside_its_workspace(lib):
    """A call that goes on to its channels-first copies writes them behind the plan's own
    workspace: the size that it asks for has to hold them."""
    copied = staged = 0
    for args in CHANNELS_LAST_CASES:
        problem = _capi.Problem.make(*args)
        ref = ctypes.byref(problem)
        x_bytes = 2 * math.prod(args[0])
        y_bytes = 2 * math.prod(out_shape(lib, problem, *args[:2]))
        plan = lib.convnd_hip_forward_workspace_size(ref, _capi.BFLOAT16)
        for layout, copies in ((_capi.CHANNELS_LAST, x_bytes + y_bytes), (_capi.CHANNELS_LAST_INPUT, x_bytes)):
            need = lib.convnd_hip_forward_workspace_size_layout(ref, _capi.BFLOAT16, layout)
            status = lib.convnd_hip_forward_layout(ref, _capi.BFLOAT16, layout, 0, NOWHERE, NOWHERE, None, NOWHERE,
                                                   NOWHERE, need, None)
            assert status == _capi.LAUNCH_FAILED
            if "channels-last input copy" in lib.convnd_hip_last_error().decode():
                assert need >= plan + copies, (args, layout)
                copied += 1
            else:
                staged += 1
    assert copied > 50 and staged > 0, (copied, staged)


# dtype, pass (0 forward, 1 input gradient), shapes: the halo of one octet in power-of-two boxes of
# 128 positions (64 from four output-channel tiles on) just does not fit LDS with its tables and pitches,
# reaches past 64 rows or 255 columns, or there are too few positions.
NO_PLAIN_PLAN = [
    ("bf16", 0, ((1, 16, 11, 11, 11, 11, 11), (32, 16, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1)),
    ("bf16", 0, ((1, 8, 9, 9, 9, 9, 9), (16, 8, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1)),
    ("bf16", 0, ((3, 48, 8, 7, 4, 8, 13), (24, 48, 3, 3, 3, 3, 3), (2,) * 5, (1,) * 5, (1,) * 5, 1)),
    ("bf16", 0, ((1, 32, 2, 3, 2, 4), (32, 32, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1)),
    ("fp32", 0, ((1, 20, 18, 12, 18, 16), (8, 5, 4, 4, 5, 3), (1, 2, 3, 1), (1, 3, 6, 1), (1, 2, 3, 1), 4)),
    ("fp32", 0, ((2, 64, 4, 9, 10, 11, 5), (1, 64, 3, 3, 3, 3, 3), (1,) * 5, (1, 2, 0, 1, 4), (2, 1, 1, 3, 3), 1)),
    ("fp32", 0, ((1, 192, 200), (64, 48, 3), (2,), (0,), (1,), 4)),
    ("fp32", 1, ((1, 2, 2, 2, 2, 2, 3, 2, 3), (16, 2, 3, 3, 2, 3, 3, 2, 3), (1,) * 7, (1, 1, 0, 1, 0, 1, 0), (1,) * 7, 1)),
]
# Just inside the same line.
PLAIN_PLAN = [
    ("bf16", 1, ((1, 2, 5, 5, 5, 5, 5, 5), (32, 2, 3, 3, 3, 3, 3, 3), (1,) * 6, (1,) * 6, (1,) * 6, 1)),
    ("bf16", 1, ((1, 96, 1, 7, 1, 3, 4, 5), (32, 96, 3, 3, 3, 3, 3, 3), (1,) * 6, (1, 0, 1, 0, 2, 1), (1,) * 6, 1)),
    ("fp32", 0, ((1, 12, 3, 5, 1, 2, 2, 2, 5), (128, 3, 3, 3, 3, 3, 1, 3, 1), (1,) * 7, (0, 2, 1, 1, 0, 1, 0), (1,) * 7, 4)),
    ("fp32", 0, ((2, 4, 2, 10, 3, 5, 11), (80, 2, 3, 3, 3, 2, 4), (2,) * 5, (1, 1, 1, 0, 1), (1,) * 5, 2)),
    ("fp32", 1, ((3, 32, 5, 5, 2, 7, 2, 2, 6), (64, 8, 3, 3, 3, 3, 1, 3, 2), (1,) * 7, (0, 0, 2, 2, 0, 1, 0), (1,) * 7, 4)),
]


@pytest.mark.parametrize(("dtype", "which", "args"), NO_PLAIN_PLAN + PLAIN_PLAN)
def test_calls_without_tables(lib, dtype, which, args):
    """Without tables, an MFMA plan whose problem has no plain plan goes on to the direct kernel
    (which such problems had before); any other fails for its tables."""
    dt = {"bf16": _capi.BFLOAT16, "fp32": _capi.FLOAT32}[dtype]
    problem = _capi.Problem.make(*args)
    ref = ctypes.byref(problem)
    assert lib.convnd_hip_plan_name(ref, dt, which) == b"mfma"
    if which == 0:
        need = lib.convnd_hip_forward_workspace_size(ref, dt)
        status = lib.convnd_hip_forward(ref, dt, NOWHERE, NOWHERE, None, NOWHERE, NOWHERE, need, None)
    else:
        need = lib.convnd_hip_backward_workspace_size(ref, dt, 1, 0, 0)
        status = lib.convnd_hip_backward(ref, dt, NOWHERE, NOWHERE, NOWHERE, NOWHERE, None, None, NOWHERE, need, None)
    assert status == _capi.LAUNCH_FAILED
    message = lib.convnd_hip_last_error().decode()
    if (dtype, which, args) in NO_PLAIN_PLAN:
        assert message.startswith("direct "), message
    else:
        assert message.startswith("geometry tables"), message


def noalloc(lib, problem, dt):
    return lib.convnd_hip_forward_noalloc(ctypes.byref(problem), dt, NOWHERE, NOWHERE, None, NOWHERE, None)


def test_noalloc_plans_a_geometry_once(lib):
    """A plan search takes milliseconds, a lookup microseconds: only the first call of a geometry
    searches, also where neither its three-part plan nor six copies fit the scratch."""
    problem = _capi.Problem.make((32, 48, 18, 17, 16, 7), (48, 48, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1)
    times = []
    for _ in range(12):
        start = time.perf_counter()
        assert noalloc(lib, problem, _capi.FLOAT32) == _capi.WORKSPACE_TOO_SMALL
        times.append(time.perf_counter() - start)
    assert min(times[1:]) < times[0] / 10, times


# Layers whose plan stages a copy larger than the scratch, while another, staged straight from the
# input, needs little (all but the last, whose packed weights alone exceed it).
@pytest.mark.parametrize(
    ("x_shape", "w_shape", "stride", "padding", "dilation", "groups", "taken"),
    [
        ((8, 128, 11, 10, 11, 10, 13), (8, 128, 3, 3, 3, 3, 3), (1,) * 5, (1,) * 5, (1,) * 5, 1, True),
        ((8, 32, 16, 13, 11, 13, 15), (8, 32, 3, 3, 3, 3, 3), (1,) * 5, (1,) * 5, (1,) * 5, 1, True),
        ((8, 40, 7, 7, 7, 7, 7, 7), (1, 40, 3, 3, 2, 3, 1, 2), (1,) * 6, (3, 1, 1, 2, 0, 0), (3, 1, 3, 2, 3, 1), 1, True),
        ((8, 64, 6, 6, 6, 6, 6, 6, 6), (192, 32, 3, 1, 3, 3, 3, 3, 1), (2,) * 7, (1, 0, 1, 1, 1, 1, 0), (1,) * 7, 2, True),
        ((1, 1024, 4, 4, 4, 4), (1024, 1024, 3, 3, 3, 3), (1,) * 4, (1,) * 4, (1,) * 4, 1, False),
    ],
)
def test_noalloc_takes_plans_that_fit_its_scratch(lib, x_shape, w_shape, stride, padding, dilation, groups, taken):
    problem = _capi.Problem.make(x_shape, w_shape, stride, padding, dilation, groups)
    need = lib.convnd_hip_forward_workspace_size(ctypes.byref(problem), _capi.BFLOAT16)
    assert need > _capi.NOALLOC_SCRATCH_BYTES
    status = noalloc(lib, problem, _capi.BFLOAT16)
    # (Taken: the call goes on to the device, which is not there.)
    assert status == (_capi.LAUNCH_FAILED if taken else _capi.WORKSPACE_TOO_SMALL)


@pytest.mark.parametrize(
    ("x_shape", "w_shape", "plan"),
    [
        ((1, 1, 6, 5, 7, 5, 5), (72, 1, 1, 1, 1, 1, 1), b"direct"),
        ((1, 1, 8, 8, 8, 8), (40, 1, 2, 1, 1, 1), b"direct"),
        ((1, 4, 4, 4, 4, 4), (60, 4, 1, 1, 1, 1), b"direct"),
        # Just more outputs, or products.
        ((1, 2, 6, 5, 7, 5, 5), (72, 2, 1, 1, 1, 1, 1), b"mfma"),
        ((1, 1, 8, 8, 8, 9), (40, 1, 2, 2, 1, 1), b"mfma"),
        ((1, 5, 4, 4, 4, 4), (60, 5, 1, 1, 1, 1), b"mfma"),
    ],
)
def test_forwards_of_a_few_products_take_one_launch(lib, x_shape, w_shape, plan):
    rank = len(x_shape) - 2
    problem = _capi.Problem.make(x_shape, w_shape, (1,) * rank, (0,) * rank, (1,) * rank, 1)
    ref = ctypes.byref(problem)
    assert lib.convnd_hip_plan_name(ref, _capi.BFLOAT16, 0) == plan
    # (The workspace is the GEMM's: with an activation, applied before the one rounding, it runs.)
    assert lib.convnd_hip_forward_workspace_size(ref, _capi.BFLOAT16) > 0
