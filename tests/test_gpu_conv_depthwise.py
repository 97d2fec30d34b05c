"""Depthwise convolutions in tiles of outputs: forward and input gradient bit for bit in the oracle's
order, the weight gradient within 1e-5 * sum|terms| (fp32 sums of under 2^14 terms in another order),
at the edges of the tiles, with unaligned operands and with values that are not finite."""

import numpy as np
import pytest
import torch

import oracle
import oxide_hip as ox
from helpers import assert_bitexact, assert_within, device_time, graph_time, host, to_dev

pytestmark = pytest.mark.gpu

# batch, channels, height, width, kernel, stride, padding
CASES = [
    (2, 3, 4, 4, 3, 1, 1),      # one tile per plane: the tensor's ends in every load
    (3, 5, 7, 9, 3, 1, 1),      # partial tiles both ways
    (3, 5, 9, 7, 5, 1, 2),
    (2, 7, 14, 14, 5, 2, 2),
    (2, 7, 13, 15, 3, 2, 1),
    (2, 3, 30, 19, 3, 2, 1),    # stride 2, more than 64 outputs
    (2, 3, 11, 12, 3, 2, 0),    # inputs that no output covers
    (2, 3, 12, 11, 5, 2, 1),
    (2, 3, 11, 11, 5, 1, 0),
    (2, 3, 6, 6, 3, 1, 3),      # padding past the kernel
    (2, 2, 6, 9, 3, 2, 4),
    (1, 4, 3, 64, 5, 1, 2),     # a kernel higher than the plane
    (40, 2, 32, 29, 5, 1, 2),   # weight sums in several blocks per channel
    (70, 3, 30, 33, 3, 2, 1),
    # the same edges in layers large enough for the tiles
    (12000, 3, 4, 4, 3, 1, 1), (1800, 5, 7, 9, 3, 1, 1), (700, 5, 9, 7, 5, 1, 2),
    (400, 7, 14, 14, 5, 2, 2), (1000, 7, 13, 15, 3, 2, 1), (800, 3, 30, 19, 3, 2, 1),
    (4500, 3, 11, 12, 3, 2, 0), (1500, 3, 12, 11, 5, 2, 1), (1400, 3, 11, 11, 5, 1, 0),
    (5200, 3, 6, 6, 3, 1, 3), (5200, 2, 6, 9, 3, 2, 4), (270, 4, 3, 64, 5, 1, 2),
    (110, 2, 32, 29, 5, 1, 2), (450, 3, 30, 33, 3, 2, 1),
    # the weight gradient's blocks of one, four and eight waves, and several chunks of images, for
    # each kernel and stride that has them
    (7, 140, 14, 13, 5, 1, 2), (16, 130, 16, 16, 5, 2, 2),
    (6, 9, 28, 28, 3, 1, 1), (16, 9, 28, 29, 3, 2, 1), (7, 9, 28, 27, 5, 1, 2),
    (12, 9, 28, 28, 5, 2, 2),
    (12, 9, 28, 28, 3, 1, 1), (24, 200, 28, 28, 3, 2, 1), (48, 3, 28, 28, 5, 1, 2),
    (22, 200, 28, 28, 5, 2, 2),
    (45, 200, 28, 28, 3, 1, 1), (74, 200, 28, 28, 3, 2, 1), (45, 200, 28, 28, 5, 1, 2),
    (74, 200, 28, 28, 5, 2, 2),
]


def _case(case):
    n, c, h, w, k, s, pad = case
    r = np.random.default_rng(n * 1000 + h * w)
    x = r.standard_normal((n, c, h, w)).astype(np.float32)
    wt = r.standard_normal((c, 1, k, k)).astype(np.float32)
    b = r.standard_normal(c).astype(np.float32)
    shape = ox.conv2d_shape(n, c, h, w, c, k, s, pad, c)
    oh, ow = ox.conv2d_output_size(shape)
    g = r.standard_normal((n, c, oh, ow)).astype(np.float32)
    return shape, x, wt, b, g


def _shifted(array, dev):
    """A copy one float past its allocation's alignment."""
    flat = torch.empty(array.size + 1, device=dev)
    out = flat[1:].view(array.shape)
    out.copy_(torch.from_numpy(array))
    return out


def _run(module, dev, case, shape, x, wt, b, g, place, addend=None):
    y = torch.full(g.shape, float("nan"), device=dev)
    dx = place(addend if addend is not None else np.full(x.shape, np.nan, np.float32), dev)
    dw = torch.full(wt.shape, float("nan"), device=dev)
    xd, wd, gd = place(x, dev), place(wt, dev), place(g, dev)
    module.conv2d_forward(shape, xd, wd, place(b, dev), y)
    if addend is None:
        module.conv2d_input_backward(shape, gd, wd, dx)
    else:
        module.conv2d_input_backward_accumulate(shape, gd, wd, dx, dx)
    module.conv2d_weight_backward(shape, gd, xd, dw)
    return host(y), host(dx), host(dw)


@pytest.mark.parametrize("place", [to_dev, _shifted], ids=["aligned", "shifted"])
@pytest.mark.parametrize("case", CASES)
def test_depthwise(module, dev, case, place):
    shape, x, wt, b, g = _case(case)
    s, pad, c = case[5], case[6], case[1]
    y, dx, dw = _run(module, dev, case, shape, x, wt, b, g, place)
    rdx, rdw, _ = oracle.conv2d_backward(g, x, wt, s, pad, c)
    assert_bitexact(y, oracle.conv2d_forward(x, wt, b, s, pad, c), "forward")
    assert_bitexact(dx, rdx, "input gradient")
    size = oracle.conv2d_backward(np.abs(g), np.abs(x), np.abs(wt), s, pad, c)[1]
    assert_within(dw, rdw, 1e-5 * size.astype(np.float64) + 1e-7, "weight gradient")
    addend = np.random.default_rng(1).standard_normal(x.shape).astype(np.float32)
    _, dx, _ = _run(module, dev, case, shape, x, wt, b, g, place, addend)
    assert_bitexact(dx, oracle.accumulate(addend, rdx), "input gradient with an addend")


@pytest.mark.parametrize("case", CASES[:10] + CASES[14:26] + [
    (6, 9, 28, 28, 3, 1, 1), (12, 9, 28, 28, 5, 2, 2), (45, 200, 28, 28, 3, 1, 1),
    (74, 200, 28, 28, 5, 2, 2)])
def test_values_that_are_not_finite(module, dev, case):
    """Infinities and NaN reach the sums whose taps they meet and no other; a zero sum that starts
    at -0 stays -0."""
    shape, x, wt, b, g = _case(case)
    s, pad, c = case[5], case[6], case[1]
    x.ravel()[::37], g.ravel()[::41] = np.inf, -np.inf
    wt.ravel()[3], wt.ravel()[11] = np.nan, np.inf
    b[-1] = -0.0
    x[:, -1], wt[-1] = 0.0, -1.0
    y, dx, dw = _run(module, dev, case, shape, x, wt, b, g, to_dev)
    rdx, rdw, _ = oracle.conv2d_backward(g, x, wt, s, pad, c)
    for got, ref in ((y, oracle.conv2d_forward(x, wt, b, s, pad, c)), (dx, rdx), (dw, rdw)):
        fine = np.isfinite(ref)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
        np.testing.assert_allclose(got[fine], ref[fine], rtol=1e-4, atol=1e-4)
    assert np.array_equal(np.signbit(y[:, -1]),
                          np.signbit(oracle.conv2d_forward(x, wt, b, s, pad, c)[:, -1]))


def test_operands_that_are_not_finite_take_no_walk_per_value(module, dev):
    """NaN weights (forward, input gradient) and gradients (weight gradient) take under seven times
    the finite operands' time (1.8, 1.8 and 4.5 measured; 10, 10 and 27 with a walk over the taps of
    each output)."""
    shape, x, wt, b, g = _case((64, 192, 28, 28, 5, 1, 2))
    xd, bd, gd, y, dx, dw = (to_dev(a, dev) for a in (x, b, g, g, x, wt))

    def times(w, grad):
        return [device_time(lambda: module.conv2d_forward(shape, xd, w, bd, y)),
                device_time(lambda: module.conv2d_input_backward(shape, gd, w, dx)),
                device_time(lambda: module.conv2d_weight_backward(shape, grad, xd, dw))]

    finite = times(to_dev(wt, dev), gd)
    nan = times(to_dev(np.full_like(wt, np.nan), dev), to_dev(np.full_like(g, np.nan), dev))
    assert all(b < 7 * a for a, b in zip(finite, nan)), (finite, nan)


def test_small_layers_keep_their_pace(module, dev):
    """A layer of a few thousand outputs has no use for tiles of them: its forward and gradients
    stay near the device's shortest launches, a ReLU's over the same tensor (1.2 to 1.5 times
    measured, 2.1 in tiles)."""
    shape, x, wt, b, g = _case((2, 39, 10, 10, 3, 1, 1))
    xd, wd, bd, gd, y, dx, dw = (to_dev(a, dev) for a in (x, wt, b, g, g, x, wt))
    relu = graph_time(lambda: module.relu(xd, dx))
    times = [graph_time(lambda: module.conv2d_forward(shape, xd, wd, bd, y)),
             graph_time(lambda: module.conv2d_input_backward(shape, gd, wd, dx)),
             graph_time(lambda: module.conv2d_weight_backward(shape, gd, xd, dw))]
    assert sum(times) < 3 * 1.75 * relu, (relu, times)
