"""Which convolutions take the kernels for large layers, by the library's own account (no GPU needed):
layers that leave a matrix-core tile or the chip mostly idle keep the kernels that are faster there,
and their sums the CPU path's order."""

import pytest

import oxide_hip as ox


def _serial(n, cin, h, w, cout, k, s, pad, forward):
    shape = ox.conv2d_shape(n, cin, h, w, cout, k, s, pad, 1)
    return ox.conv2d_forward_serial(shape) if forward else ox.conv2d_input_backward_serial(shape)


# batch, in, height, width, out, kernel, stride, padding
@pytest.mark.parametrize("case,serial", [
    ((32, 64, 112, 112, 1, 3, 1, 1), True),      # a one-channel prediction head
    ((32, 64, 112, 112, 2, 5, 1, 2), True),
    ((32, 64, 112, 112, 4, 3, 1, 1), False),
    ((1, 64, 28, 28, 64, 3, 1, 1), True),        # one image: half of the chip's waves
    ((1, 64, 56, 56, 64, 3, 1, 1), False),
    ((3, 97, 15, 63, 15, 3, 1, 1), True),
    ((1024, 64, 14, 14, 4, 3, 1, 1), True),      # a per-image kernel, over 2^27 products
    ((1024, 64, 14, 14, 6, 3, 1, 1), False),
    ((1024, 16, 16, 16, 8, 5, 1, 2), True),
    ((1024, 16, 16, 16, 12, 5, 1, 2), False),
    ((26, 2, 102, 1, 12, 1, 2, 0), True),        # a strided 1 x 1 of few values
    ((16, 96, 32, 31, 64, 1, 2, 0), False),
    ((32, 64, 56, 56, 64, 3, 1, 1), False),
    ((32, 3, 224, 224, 32, 3, 2, 1), False),
])
def test_forward(case, serial):
    assert _serial(*case, forward=True) == serial


@pytest.mark.parametrize("case,serial", [
    ((32, 1, 112, 112, 64, 3, 1, 1), True),      # the gradient of a one-channel image
    ((32, 1, 112, 112, 64, 5, 1, 2), True),
    ((32, 6, 112, 112, 64, 3, 1, 1), False),
    ((1, 32, 40, 40, 32, 3, 1, 1), True),
    ((8, 1, 56, 56, 64, 3, 2, 1), True),
    ((1, 152, 11, 32, 367, 3, 2, 0), True),
    ((1024, 4, 16, 16, 16, 5, 1, 2), True),
    ((8, 33, 62, 61, 65, 3, 2, 1), False),
    ((32, 64, 56, 56, 64, 3, 1, 1), False),
    ((32, 32, 112, 112, 32, 3, 2, 1), False),
])
def test_input_gradient(case, serial):
    assert _serial(*case, forward=False) == serial


# 1 x 1 layers: batch, in, height, width, out
@pytest.mark.parametrize("case,forward,backward", [
    ((1, 128, 14, 14, 128), True, True),         # a few waves' worth of products
    ((1, 32, 64, 64, 16), True, True),
    ((4, 64, 28, 28, 64), False, True),          # a backward whose gradients share a launch
    ((1, 64, 56, 56, 64), False, True),
    ((79, 4, 44, 44, 1), False, False),          # few channels, many positions
    ((8, 64, 56, 56, 64), False, False),
    ((64, 64, 56, 56, 192), False, False),
])
def test_pointwise(case, forward, backward):
    assert _serial(*case, 1, 1, 0, forward=True) == forward
    assert _serial(*case, 1, 1, 0, forward=False) == backward


# batch, in, height, width, out, kernel, stride, padding
@pytest.mark.parametrize("case,partials,bias", [
    ((77, 576, 19, 19, 1, 3, 1, 1), 77, False),    # one output channel: a chunk per image
    ((120, 220, 7, 7, 1, 3, 1, 0), 120, False),
    ((62, 466, 6, 6, 3, 3, 2, 1), 62, False),
    ((64, 3, 28, 28, 128, 3, 2, 1), 64, True),     # few columns: an image's sums in LDS
    ((64, 1, 28, 28, 128, 3, 2, 1), 64, True),
])
def test_weight_gradient_of_few_rows_or_columns(case, partials, bias):
    """The partial sums that the workspace holds are those of the kernels of one weight per thread
    and of one image in LDS (with the bias sums)."""
    n, cin, h, w, cout, k, s, pad = case
    shape = ox.conv2d_shape(n, cin, h, w, cout, k, s, pad, 1)
    sums = cout * cin * k * k + (cout if bias else 0)
    assert ox.conv2d_workspace_size(shape) // (4 * sums) == partials
