"""Inference programs run whole (BatchNorm and the op behind it in one launch) against their
launch groups run one by one: every node's value bit for bit."""

import numpy as np
import pytest
import torch

import nn
import tensor as tn
from helpers import host

pytestmark = pytest.mark.gpu


def _norm(channels, r):
    bn = nn.BatchNorm2d(channels)
    bn.set_training(False)
    dev = bn.weight.data.device
    for t, low, high in ((bn.weight.data, 0.5, 1.5), (bn.bias.data, -0.5, 0.5),
                         (bn.state.running_mean, -0.3, 0.3),
                         (bn.state.running_variance, 0.5, 2.0)):
        t.copy_(torch.from_numpy(r.uniform(low, high, channels).astype(np.float32)).to(dev))
    return bn


@pytest.mark.parametrize("height,width", [(6, 6), (5, 7), (1, 1), (40, 52)])
def test_whole_program_equals_its_groups(dev, height, width):
    """A ReLU behind, an addition behind (either operand order), nothing behind, a BatchNorm with
    both, an addition whose other operand comes later, and one of a value to itself."""
    r = np.random.default_rng(height * width)
    c = 5
    x = tn.input((3, c, height, width))
    norms = [_norm(c, r) for _ in range(6)]
    a = norms[0](x)
    b = a.relu()
    d = norms[1](nn.Conv2d(c, c, 1)(b))
    e = b.add(d)                    # the other operand first, and before the BatchNorm
    f = norms[2](e)
    g = f.mul(e)                    # nothing to take in
    h = norms[3](g)
    i, j = h.relu(), h.add(e)       # both: the ReLU goes along
    k = norms[4](j)
    m = k.add(nn.Conv2d(c, c, 1)(i))  # the convolution runs after the BatchNorm
    o = norms[5](m)
    out = o.add(o)
    nodes = [a, b, d, e, f, g, h, i, j, k, m, o, out]
    program = tn.forward_program(out, [x])
    program.feed(x, r.standard_normal((3, c, height, width)).astype(np.float32))
    kinds = [op.kind for op in program.ops]
    assert kinds.count("batch_norm2d_eval_forward") == 6
    for op in program.ops:
        op.launch()
    program.synchronize()
    one_by_one = [program.value(t).host() for t in nodes]
    for t in nodes:
        program.value(t).copy_from(np.full(t.shape, np.nan, np.float32))
    program.run()
    program.synchronize()
    whole = [program.value(t).host() for t in nodes]
    program.capture()
    for t in nodes:
        program.value(t).copy_from(np.full(t.shape, np.nan, np.float32))
    program.replay()
    program.synchronize()
    replayed = [program.value(t).host() for t in nodes]
    for t, p, q, s in zip(nodes, one_by_one, whole, replayed):
        assert np.isfinite(p).all()
        assert np.array_equal(p, q) and np.array_equal(p, s), t


@pytest.mark.parametrize("shape", [
    (1, 4, 1, 5),    # the smallest plane a unit can leave
    (4, 1, 3, 3),    # one channel: the next plane's channel is the same
    (2, 6, 7, 7),    # a unit may start one to three values before a plane's end
    (3, 4, 3, 5),    # planes of 4 n + 3 values
    (1, 4, 3, 7),    # one image: every plane's inverse deviation is stored
    (64, 96, 7, 7),  # many blocks
    (3, 5, 5, 7),    # no whole number of units: value by value
])
def test_planes_of_no_whole_units(dev, shape):
    """Units of four values that may reach into the next plane: nothing, a ReLU and an addition
    behind, against the groups one by one."""
    r = np.random.default_rng(sum(shape))
    x = tn.input(shape)
    a = _norm(shape[1], r)(x)
    b = a.relu()
    d = _norm(shape[1], r)(b)
    e = d.add(a)
    f = _norm(shape[1], r)(e)
    program = tn.forward_program(f.mul(e), [x])
    program.feed(x, r.standard_normal(shape).astype(np.float32))
    for op in program.ops:
        op.launch()
    program.synchronize()
    nodes = [a, b, d, e, f]
    one_by_one = [program.value(t).host() for t in nodes]
    for t in nodes:
        program.value(t).copy_from(np.full(t.shape, np.nan, np.float32))
    program.run()
    program.synchronize()
    for t, want in zip(nodes, one_by_one):
        assert np.isfinite(want).all()
        assert np.array_equal(program.value(t).host(), want), t


class _Buffer:
    """A program's buffer as torch takes it in."""

    def __init__(self, view):
        self.__cuda_array_interface__ = {"data": (view.ptr, False), "typestr": "<f4",
                                         "shape": tuple(view.shape), "strides": None,
                                         "version": 2}


def test_tensors_past_32_bit_indexes(dev):
    """2^31 values and more in planes of no whole float4: past the joined kernel's indexes, so its
    launches one by one."""
    shape = (1, 3, 26755, 26755)
    x = tn.input(shape)
    norm = _norm(3, np.random.default_rng(1))
    a = norm(x)
    b = a.relu()
    program = tn.forward_program(b, [x])
    xs, ys, zs = (torch.as_tensor(_Buffer(program.value(t)), device=dev).view(-1)
                  for t in (x, a, b))
    assert xs.numel() >= 1 << 31 and xs.numel() % 4 != 0
    xs.normal_()
    ys.fill_(float("nan"))
    zs.fill_(float("nan"))
    torch.cuda.synchronize()
    program.run()
    program.synchronize()
    mean, variance = norm.state.running_mean, norm.state.running_variance
    inverse = 1 / torch.sqrt(variance + 1e-5)
    for start, c in ((0, 0), ((1 << 31) - (1 << 20), 2), (xs.numel() - (1 << 20), 2)):
        v, y, z = (t[start:start + (1 << 20)] for t in (xs, ys, zs))
        want = (v - mean[c]) * inverse[c] * norm.weight.data[c] + norm.bias.data[c]
        assert torch.allclose(y, want, rtol=1e-6, atol=1e-6)  # a rounding in the square root
        assert torch.equal(z, y.relu())
    assert bool(zs.isfinite().all())


@pytest.mark.parametrize("shape", [(3, 5, 6, 6), (2, 6, 7, 7), (1, 4, 3, 7), (64, 96, 7, 7),
                                   (3, 5, 5, 7), (3, 5, 1, 1)])
def test_inverse_deviations_and_values_that_are_not_finite(dev, shape):
    """Infinities and NaN among the input and the running statistics, nothing, a ReLU (whose NaN is
    0) and an addition behind: values and stored inverse deviations as the groups one by one leave
    them, after a run and after replays with eager runs between."""
    r = np.random.default_rng(sum(shape))
    x = tn.input(shape)
    norms = [_norm(shape[1], r) for _ in range(3)]
    for norm, bad in zip(norms, (np.inf, np.nan, -2.0)):  # the last: a NaN square root
        norm.state.running_variance[shape[1] - 2:shape[1] - 1] = bad
    a = norms[0](x)
    b = a.relu()
    d = norms[1](b)
    e = d.add(a)
    f = norms[2](e)
    program = tn.forward_program(f.mul(e), [x])
    values = r.standard_normal(shape).astype(np.float32)
    values.ravel()[1::19], values.ravel()[2::23], values.ravel()[3::29] = np.inf, np.nan, -np.inf
    program.feed(x, values)
    for op in program.ops:
        op.launch()
    program.synchronize()
    groups = [op for op in program.ops if op.kind == "batch_norm2d_eval_forward"]
    views = [program.value(t) for t in (a, b, d, e, f)] + [g.writes["inverse_std"] for g in groups]
    assert len(views) == 8
    want = [v.host() for v in views]
    assert np.isnan(want[0]).any() and not np.isnan(want[1]).any()

    def same(start):
        for v in views:
            v.copy_from(np.full(v.shape, 7.0, np.float32))
        start()
        program.synchronize()
        return all(np.array_equal(v.host(), w, equal_nan=True) for v, w in zip(views, want))

    assert same(program.run)
    program.capture()
    assert same(program.replay) and same(program.run) and same(program.replay)
