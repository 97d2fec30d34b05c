"""Convolutions over planes too large for the per-image kernels, on the matrix cores: forward,
input gradient (with an addend) and weight / bias gradients against the oracle at the edges of
their tiles (32 rows, 32 positions, channel pairs), within 1e-5 * sum|terms|: an fp32 sum of n
terms in any order is off by at most n * 2^-24 * sum|terms|, and by about sqrt(n) * 2^-24 of it
in practice, under 1e-5 for every n below 2^14."""

import numpy as np
import pytest
import torch

import oracle
import oxide_hip as ox
from helpers import (assert_conv_forward, assert_conv_input_gradient, assert_within, device_time,
                     host, to_dev)

pytestmark = pytest.mark.gpu

# batch, in, height, width, out, kernel, stride, padding
CASES = [
    (40, 3, 75, 73, 33, 3, 2, 1),     # a stem: one and a half channel pairs, 33 output rows
    (6, 32, 33, 31, 32, 3, 1, 1),     # one row tile, odd planes, positions across images
    (6, 17, 40, 29, 70, 3, 1, 1),     # an odd channel, 64 + 6 rows
    (1, 64, 65, 66, 64, 3, 1, 1),     # whole tiles
    (8, 40, 30, 34, 96, 3, 2, 1),
    (4, 24, 41, 37, 40, 5, 1, 2),
    (12, 10, 61, 43, 24, 5, 2, 2),
    (2, 96, 32, 31, 64, 1, 2, 0),     # a strided 1 x 1: three of four inputs feed no output
    (14, 20, 33, 33, 20, 3, 1, 0),    # no padding
    (16, 70, 35, 20, 16, 3, 2, 0),
    (1, 24, 35, 33, 20, 1, 1, 1),     # a padded 1 x 1
    (20, 48, 17, 16, 66, 3, 1, 1),    # planes a per-image kernel holds, over 2^27 products
    (60, 64, 15, 14, 144, 3, 2, 1),
    (12, 64, 3, 300, 64, 3, 1, 0),    # one output row a plane
    (12, 61, 5, 300, 65, 3, 2, 0),    # two
    (16, 24, 64, 63, 6, 3, 1, 1),     # six channels in a tile of 32
    (16, 6, 64, 63, 24, 3, 1, 1),
]


def _case(case, dev):
    n, cin, h, w, cout, k, s, pad = case
    r = np.random.default_rng(abs(hash(case)) & 0xFFFFFFFF)
    x = r.standard_normal((n, cin, h, w)).astype(np.float32)
    wt = (r.standard_normal((cout, cin, k, k)) * 0.3).astype(np.float32)
    b = r.standard_normal(cout).astype(np.float32)
    shape = ox.conv2d_shape(n, cin, h, w, cout, k, s, pad, 1)
    oh, ow = ox.conv2d_output_size(shape)
    g = r.standard_normal((n, cout, oh, ow)).astype(np.float32)
    return shape, x, wt, b, g


@pytest.mark.parametrize("case", CASES)
def test_forward(module, dev, case):
    shape, x, wt, b, g = _case(case, dev)
    y = torch.full(g.shape, float("nan"), device=dev)
    module.conv2d_forward(shape, to_dev(x, dev), to_dev(wt, dev), to_dev(b, dev), y)
    assert not ox.conv2d_forward_serial(shape)
    assert_conv_forward(host(y), x, wt, b, case[6], case[7], 1, "forward")


@pytest.mark.parametrize("addend", ["none", "separate", "in place"])
@pytest.mark.parametrize("case", CASES)
def test_input_gradient(module, dev, case, addend):
    shape, x, wt, _, g = _case(case, dev)
    gd, wd = to_dev(g, dev), to_dev(wt, dev)
    dx = torch.full(x.shape, float("nan"), device=dev)
    if addend == "none":
        module.conv2d_input_backward(shape, gd, wd, dx)
    elif addend == "separate":
        module.conv2d_input_backward_accumulate(shape, gd, wd, to_dev(x, dev), dx)
    else:
        dx = to_dev(x, dev)
        module.conv2d_input_backward_accumulate(shape, gd, wd, dx, dx)
    assert not ox.conv2d_input_backward_serial(shape)
    assert_conv_input_gradient(host(dx), g, wt, case[6], case[7], 1, x.shape,
                               None if addend == "none" else x, "input gradient")


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("case", [(8, 33, 34, 31, 40, 3, 1, 1), (8, 30, 40, 44, 66, 3, 2, 1)])
def test_weights_that_are_not_finite(module, dev, case, value):
    """An infinite or NaN weight reaches the outputs whose tap lies inside the input, and no
    other: taps outside are skipped, as the CPU path skips them."""
    shape, x, wt, b, g = _case(case, dev)
    wt[3, 5, 0, 0] = value
    y = torch.empty(g.shape, device=dev)
    dx = torch.empty(x.shape, device=dev)
    module.conv2d_forward(shape, to_dev(x, dev), to_dev(wt, dev), to_dev(b, dev), y)
    module.conv2d_input_backward(shape, to_dev(g, dev), to_dev(wt, dev), dx)
    ref_y = oracle.conv2d_forward(x, wt, b, case[6], case[7], 1)
    ref_dx = oracle.conv2d_backward(g, x, wt, case[6], case[7], 1)[0]
    for got, ref in ((host(y), ref_y), (host(dx), ref_dx)):
        fine = np.isfinite(ref)
        assert 0 < fine.sum() < ref.size
        assert np.array_equal(fine, np.isfinite(got))
        np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-4, atol=1e-4)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])


# batch, in, height, width, out, kernel, stride, padding: one to nine column tiles per block, one
# and two row tiles, groups of one row and of several, image ends inside a group, widths padded
# to eight positions, one partial sum
WEIGHT_CASES = CASES + [
    (1, 130, 9, 11, 33, 3, 1, 1),
    (3, 64, 45, 44, 64, 3, 1, 1),
    (2, 18, 50, 47, 40, 7, 3, 2),
    (1, 2, 3, 300, 5, 3, 1, 1),
    (40, 24, 3, 120, 33, 3, 1, 0),    # one output row, two
    (40, 24, 4, 120, 33, 3, 1, 0),
    (4, 8, 18, 18, 32, 3, 1, 1),      # planes an LDS plan holds, over 64 positions
]


@pytest.mark.parametrize("case", WEIGHT_CASES)
def test_weight_gradient(module, dev, case):
    shape, x, wt, _, g = _case(case, dev)
    dw = torch.full(wt.shape, float("nan"), device=dev)
    module.conv2d_weight_backward(shape, to_dev(g, dev), to_dev(x, dev), dw)
    ref = oracle.conv2d_backward(g, x, wt, case[6], case[7], 1)[1]
    size = oracle.conv2d_backward(np.abs(g), np.abs(x), np.abs(wt), case[6], case[7], 1)[1]
    assert_within(host(dw), ref, 1e-5 * size.astype(np.float64) + 1e-7, "weight gradient")


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("case", [(8, 33, 34, 31, 40, 3, 1, 1), (8, 30, 40, 44, 66, 3, 2, 1)])
def test_gradients_that_are_not_finite(module, dev, case, value):
    """An infinite or NaN output gradient in a corner reaches the weights whose tap lies inside
    the input there, and no other."""
    shape, x, wt, _, g = _case(case, dev)
    g[0, 4, 0, 0] = value
    dw = torch.empty(wt.shape, device=dev)
    module.conv2d_weight_backward(shape, to_dev(g, dev), to_dev(x, dev), dw)
    ref = oracle.conv2d_backward(g, x, wt, case[6], case[7], 1)[1]
    fine = np.isfinite(ref)
    assert (~fine).sum() == 4 * case[1]  # the corner's four taps of one output channel
    assert np.array_equal(np.isnan(ref), np.isnan(host(dw)))
    assert np.array_equal(host(dw)[np.isinf(ref)], ref[np.isinf(ref)])
    np.testing.assert_allclose(host(dw)[fine], ref[fine], rtol=1e-3, atol=1e-3)


# every kernel's other pass: both 5 x 5 forms, 3 x 3, strided and padded 1 x 1; odd planes, channels
# of no whole pairs, rows of no whole tiles
NOT_FINITE = [
    (8, 6, 56, 55, 24, 5, 1, 2), (8, 25, 57, 55, 40, 5, 2, 2), (8, 21, 61, 62, 40, 3, 1, 1),
    (8, 33, 62, 61, 65, 3, 2, 1), (16, 96, 32, 31, 64, 1, 2, 0), (9, 24, 35, 33, 20, 1, 1, 1),
]


def _assert_alike(got, ref):
    fine = np.isfinite(ref)
    assert 0 < (~fine).sum() and np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("case", NOT_FINITE)
def test_operands_that_are_not_finite_in_every_kernel(module, dev, case):
    """Corner taps infinite and NaN (in the forward an output channel all NaN too), the input
    gradient added in place; corners and a value inside of the output gradient infinite and NaN."""
    n, cin, h, w, cout, k, s, pad = case
    shape, x, wt, b, g = _case(case, dev)
    bad = wt.copy()
    bad[3, 5, 0, 0], bad[7, 2, -1, -1] = np.inf, np.nan
    y, dx = torch.empty(g.shape, device=dev), to_dev(x, dev)
    module.conv2d_input_backward_accumulate(shape, to_dev(g, dev), to_dev(bad, dev), dx, dx)
    ref = oracle.conv2d_backward(g, x, bad, s, pad, 1)[0]
    _assert_alike(host(dx), oracle.accumulate(x, ref))
    bad[cout - 1] = np.nan
    module.conv2d_forward(shape, to_dev(x, dev), to_dev(bad, dev), to_dev(b, dev), y)
    _assert_alike(host(y), oracle.conv2d_forward(x, bad, b, s, pad, 1))
    g[0, 1, 0, 0], g[1, 2, -1, -1], g[n - 1, 3, 0, -1] = -np.inf, np.nan, np.inf
    g[2, 4, g.shape[2] // 2, 1] = np.nan
    dw = torch.empty(wt.shape, device=dev)
    module.conv2d_weight_backward(shape, to_dev(g, dev), to_dev(x, dev), dw)
    _assert_alike(host(dw), oracle.conv2d_backward(g, x, wt, s, pad, 1)[1])


def test_operands_that_are_not_finite_take_no_walk_per_value(module, dev):
    """A network whose values have left the finite range keeps about its pace: under eight times the
    finite operands' time (forward and input gradient 3.3, weight gradient 3.7, measured), where a
    serial walk over each sum takes 35 times."""
    shape, x, wt, b, g = _case((8, 64, 28, 28, 64, 5, 1, 2), dev)
    xd, bd, gd, y, dx, dw = (to_dev(a, dev) for a in (x, b, g, g, x, wt))

    def times(w, grad):
        return [device_time(lambda: module.conv2d_forward(shape, xd, w, bd, y)),
                device_time(lambda: module.conv2d_input_backward(shape, gd, w, dx)),
                device_time(lambda: module.conv2d_weight_backward(shape, grad, xd, dw))]

    finite = times(to_dev(wt, dev), gd)
    nan = times(to_dev(np.full_like(wt, np.nan), dev), to_dev(np.full_like(g, np.nan), dev))
    assert all(b < 8 * a for a, b in zip(finite, nan)), (finite, nan)


@pytest.mark.parametrize("batch,channels,height,width", [
    (1, 3, 64, 64),      # the most terms a wave sums
    (1, 3, 63, 67),      # a block per channel, scalar loads
    (5, 7, 60, 56),      # float4s, a last round that is not full
    (300, 33, 8, 8),     # many short planes
])
def test_bias_gradient(module, dev, batch, channels, height, width):
    r = np.random.default_rng(batch)
    g = r.standard_normal((batch, channels, height, width)).astype(np.float32)
    shape = ox.conv2d_shape(batch, 2, height, width, channels, 3, 1, 1, 1)
    db = torch.full((channels,), float("nan"), device=dev)
    flat = torch.empty(g.size + 1, device=dev)
    for lead in (0, 1):  # aligned, and one float past it
        gd = flat[lead:lead + g.size].view(g.shape)
        gd.copy_(torch.from_numpy(g))
        module.conv2d_bias_backward(shape, gd, db)
        assert_within(host(db), g.astype(np.float64).sum((0, 2, 3)),
                      1e-5 * np.abs(g).astype(np.float64).sum((0, 2, 3)), "bias gradient")


def test_paired_backward_leaves_wide_bias_sums_to_their_kernel(module, dev):
    """A 1 x 1 backward whose two products share a launch, with more bias terms than a wave sums:
    the bias equals the separate entry point's, bit for bit."""
    r = np.random.default_rng(5)
    shape = ox.conv2d_shape(150, 16, 7, 7, 16, 1, 1, 0, 1)
    x = to_dev(r.standard_normal((150, 16, 7, 7)).astype(np.float32), dev)
    g = to_dev(r.standard_normal((150, 16, 7, 7)).astype(np.float32), dev)
    wt = to_dev(r.standard_normal((16, 16, 1, 1)).astype(np.float32), dev)
    dx, dw = torch.empty_like(x), torch.empty_like(wt)
    db, ref = (torch.full((16,), float("nan"), device=dev) for _ in range(2))
    module.conv2d_backward(shape, g, x, wt, dx, dw, db)
    module.conv2d_bias_backward(shape, g, ref)
    assert np.array_equal(host(db), host(ref))
    assert_within(host(db), host(g).astype(np.float64).sum((0, 2, 3)),
                  1e-5 * np.abs(host(g)).astype(np.float64).sum((0, 2, 3)), "bias gradient")


# 1 x 1 layers, batch, in, height, width, out: pairs of positions (even planes, two blocks per
# CU), single ones (odd planes; few blocks), four waves per position; ragged rows, positions
# and channel chunks (16, 32 and 128 channels); a plane of 64 in a layer of over 2^27 products
POINTWISE = [
    (15, 37, 60, 150, 33), (16, 40, 93, 91, 70), (36, 33, 31, 13, 50), (66, 129, 11, 9, 40),
    (200, 70, 9, 9, 5), (23, 200, 13, 6, 96), (9, 400, 10, 8, 130), (40, 130, 8, 8, 416),
]


@pytest.mark.parametrize("case", POINTWISE)
@pytest.mark.parametrize("lead", [0, 1])
def test_pointwise(module, dev, case, lead):
    """Forward, input gradient and the input gradient added in place; with tensors one float past
    their allocation's alignment (lead 1) too."""
    n, cin, h, w, cout = case
    r = np.random.default_rng(cin * cout + lead)
    shape = ox.conv2d_shape(n, cin, h, w, cout, 1, 1, 0, 1)
    assert not ox.conv2d_forward_serial(shape) and not ox.conv2d_input_backward_serial(shape)

    def device(a):
        flat = torch.empty(a.size + lead, device=dev)[lead:].view(a.shape)
        return flat.copy_(torch.from_numpy(a))

    x = r.standard_normal((n, cin, h, w)).astype(np.float32)
    wt = (r.standard_normal((cout, cin, 1, 1)) * 0.3).astype(np.float32)
    b = r.standard_normal(cout).astype(np.float32)
    g = r.standard_normal((n, cout, h, w)).astype(np.float32)
    xd, wd, gd = device(x), device(wt), device(g)
    y, dx, summed = device(np.full_like(g, np.nan)), device(np.full_like(x, np.nan)), device(x)
    module.conv2d_forward(shape, xd, wd, device(b), y)
    module.conv2d_input_backward(shape, gd, wd, dx)
    module.conv2d_input_backward_accumulate(shape, gd, wd, summed, summed)
    matrix = wt.reshape(cout, cin).astype(np.float64)
    for got, m, v, add in ((y, matrix, x, b[:, None, None]), (dx, matrix.T, g, 0.0),
                           (summed, matrix.T, g, x)):
        flat = v.reshape(n, v.shape[1], -1).astype(np.float64)
        shaped = (n, m.shape[0], h, w)
        ref = (m @ flat).reshape(shaped) + add
        size = (np.abs(m) @ np.abs(flat)).reshape(shaped) + np.abs(add)
        assert_within(host(got), ref, 1e-5 * size, "1 x 1")
