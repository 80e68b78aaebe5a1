"""Precision of fp32 layers that run on bf16 parts where fp32 products of the direct kernels served
before (marked ``gpu``): no larger error against float64 than those products' sums have.

A sum of n products added one by one, each addition rounded to fp32, has a relative error
(2-norm over many outputs) of about r * sqrt(n / 2) for terms of zero mean and r * sqrt(n / 3)
for terms of one sign, with r = 2^-23.5 / sqrt(12), the root mean square of one rounding: the
partial sum at step k carries sqrt(k / n) or k / n of the result. Six truncated part products
in one accumulator are ten times further off on same-sign data (1.4e-5 against 1.1e-6 at
n = 7776) and twice as far on sparse data.
"""

import ctypes
import math

import pytest
import torch

import helpers
from torch_convnd import _build, _capi, conv_nd, load_native

pytestmark = pytest.mark.gpu

ROUNDING = 2.0**-23.5 / math.sqrt(12.0)
SPARSE = 0.004  # share of non-zero inputs

# x shape, w shape, stride, passes on eight products (y, dx, dw), operand layout of the forward
CASES = {
    "wide": ((1, 72, 4, 4, 4, 5), (80, 72, 3, 3, 3, 3), 1, ("y", "dx"), 3),
    "few_positions": ((1, 32, 2, 3, 2, 4), (33, 32, 3, 3, 3, 3), 1, ("y", "dx"), 3),
    "strided_rank5": ((1, 16, 7, 7, 7, 7, 9), (40, 16, 3, 3, 3, 3, 3), 2, ("y",), 3),
    # The planes of three parts fit LDS in no box: copies of the channels, whole octets or not.
    "copies": ((1, 8, 4, 4, 4, 4, 5, 6), (14, 8, 3, 3, 3, 3, 3, 3), 2, ("y",), 1),
    "copies_odd": ((2, 3, 4, 5, 4, 5, 4, 5), (8, 3, 3, 3, 3, 3, 3, 3), 2, ("y",), 1),
}


@pytest.fixture(scope="module", autouse=True)
def native():
    load_native()


def draw(kind, shape, generator):
    if kind == "same_sign":
        return torch.rand(shape, generator=generator) + 2.0**-20
    x = torch.randn(shape, generator=generator)
    if kind == "sparse":
        x = torch.where(torch.rand(shape, generator=generator) < SPARSE, x, torch.zeros(()))
    return x


def bound(kind, n):
    """One rounding of the result at least, and a tenth for the scatter of the estimate."""
    terms = n / 3 if kind == "same_sign" else (SPARSE * n if kind == "sparse" else n) / 2
    return 1.1 * ROUNDING * math.sqrt(terms + 1)


@pytest.mark.parametrize("kind", ["dense", "same_sign", "sparse"])
@pytest.mark.parametrize("name", list(CASES))
def test_split_products_are_no_further_off_than_fp32_products(name, kind):
    x_shape, w_shape, stride, passes, parts = CASES[name]
    rank = len(x_shape) - 2
    args = ((stride,) * rank, (1,) * rank, (1,) * rank, 1)
    print(f"[precision] {name} {kind} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    assert lib.convnd_hip_plan_check(ctypes.byref(_capi.Problem.make(x_shape, w_shape, *args)),
                                     _capi.FLOAT32) == _capi.SUCCESS
    plans = dict(zip(("y", "dx", "dw"), _capi.plan_details(lib, x_shape, w_shape, *args, torch.float32)))
    assert plans["y"]["parts"] == parts, plans["y"]
    for p in passes:
        assert plans[p].get("products") == 8 or (p == "dw" and plans[p]["kernel"] == "mfma_wgrad_cm"), plans[p]
    g = torch.Generator().manual_seed(81)
    x = draw(kind, x_shape, g)
    w = draw("same_sign" if kind == "same_sign" else "dense", w_shape, g)
    ref_y = helpers.oracle_forward(x, w, None, *args)
    dy = draw(kind, ref_y.shape, g)
    ref_dx, ref_dw, _ = helpers.oracle_backward(dy, x, w, *args)
    dev = [t.cuda().requires_grad_() for t in (x, w)]
    y = conv_nd(dev[0], dev[1], None, *args, backend="native")
    dx, dw = torch.autograd.grad(y, dev, dy.cuda())
    taps = math.prod(w_shape[2:])
    for p, got, ref, n in (("y", y, ref_y, w_shape[1] * taps), ("dx", dx, ref_dx, w_shape[0] * taps)):
        if p in passes:
            error = ((got.detach().double().cpu() - ref).norm() / ref.norm()).item()
            assert error <= bound(kind, n), (p, error, bound(kind, n))


# Strided last axes whose halo only the channel-major weight gradient holds.
WEIGHT_CASES = {
    "small": ((1, 16, 7, 7, 7, 7, 9), (8, 16, 3, 3, 3, 3, 3)),
    "ragged": ((2, 8, 9, 7, 7, 7, 5), (24, 8, 3, 3, 3, 3, 3)),
    "many_boxes": ((2, 8, 11, 11, 9, 9, 9), (16, 8, 3, 3, 3, 3, 3)),
}


def weight_bound(kind, positions):
    """Position i in thread i mod 256, then a tree of eight levels, whose partial sums carry
    1 (zero mean) or 2^-level (one sign) of the squared result together."""
    chain = positions / 256
    if kind == "same_sign":
        terms = chain / 768 + 2
    else:
        share = SPARSE if kind == "sparse" else 1.0
        terms = share * chain / 2 + min(8, share * positions)
    return 1.1 * ROUNDING * math.sqrt(terms + 1)


@pytest.mark.parametrize("kind", ["dense", "same_sign", "sparse"])
@pytest.mark.parametrize("name", list(WEIGHT_CASES))
def test_strided_weight_gradient_is_no_further_off_than_fp32_products(name, kind):
    x_shape, w_shape = WEIGHT_CASES[name]
    args = ((2,) * 5, (1,) * 5, (1,) * 5, 1)
    print(f"[precision] weight gradient {name} {kind} x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    assert lib.convnd_hip_plan_check(ctypes.byref(_capi.Problem.make(x_shape, w_shape, *args)),
                                     _capi.FLOAT32) == _capi.SUCCESS
    assert _capi.plan_details(lib, x_shape, w_shape, *args, torch.float32)[2]["kernel"] == "mfma_wgrad_cm"
    g = torch.Generator().manual_seed(82)
    x = draw(kind, x_shape, g)
    w = draw("dense", w_shape, g)
    out = tuple((n - 1) // 2 + 1 for n in x_shape[2:])
    dy = draw("dense" if kind == "sparse" else kind, (x_shape[0], w_shape[0], *out), g)
    ref = helpers.oracle_backward(dy, x, w, *args)[1]
    dev = [t.cuda().requires_grad_() for t in (x, w)]
    y = conv_nd(dev[0], dev[1], None, *args, backend="native")
    dw = torch.autograd.grad(y, dev[1], dy.cuda())[0]
    error = ((dw.double().cpu() - ref).norm() / ref.norm()).item()
    assert error <= weight_bound(kind, x_shape[0] * math.prod(out)), (error, weight_bound(kind, x_shape[0] * math.prod(out)))


def test_long_chunks_add_the_small_products_first():
    """Six products of a unit-stride weight gradient in long position chunks: the roundings of the
    large product's K steps (the last sixth of the items), not those of all. What the truncated
    parts drop, up to 2^-21 of a product and about 2^-24 of it in the mean, is added."""
    x_shape, w_shape = (2, 112, 8, 6, 7, 6, 5), (3, 112, 3, 3, 3, 3, 3)
    args = ((1,) * 5, (1,) * 5, (1,) * 5, 1)
    print(f"[precision] long chunks x={x_shape} w={w_shape}", flush=True)
    lib = _build.hip_library()
    plan = _capi.plan_details(lib, x_shape, w_shape, *args, torch.float32)[2]
    assert plan["kernel"] == "mfma_wgrad_cm" and plan["items_per_pc"] > plan["items"] / 6, plan
    g = torch.Generator().manual_seed(83)
    x, w = torch.randn(x_shape, generator=g), torch.randn(w_shape, generator=g)
    dy = torch.randn((2, 3, *x_shape[2:]), generator=g)
    ref = helpers.oracle_backward(dy, x, w, *args)[1]
    dev = [t.cuda().requires_grad_() for t in (x, w)]
    dw = torch.autograd.grad(conv_nd(dev[0], dev[1], None, *args, backend="native"), dev[1], dy.cuda())[0]
    error = ((dw.double().cpu() - ref).norm() / ref.norm()).item()
    # Eight K steps an item, four in each of two sums with eight waves; the MFMA adds a step's 32
    # products to the sum in up to four parts, each rounded.
    roundings = 4 * plan["items"] / 6 * (8 if plan["waves"] == 4 else 4)
    bound = 1.1 * math.hypot(ROUNDING * math.sqrt(roundings / 2 + plan["npc"]), 2.0**-24)
    print(f"error {error:.2e} bound {bound:.2e}", flush=True)
    assert error <= bound, (error, bound)
