"""BatchNorm training forward and backward with one block per channel over planes of 64 values and
more, against the oracle at the edges of its units (planes of 4 n + 0 .. 3 values, one to eight
units per thread, 256 and 1024 threads, the shapes just past them)."""

import numpy as np
import pytest
import torch

import oracle
import oxide_hip as ox
from helpers import (assert_within, check_batch_norm_backward, check_batch_norm_forward, host,
                     to_dev)

pytestmark = pytest.mark.gpu

SHAPES = [
    (2, 3, 8, 8),       # the smallest plane
    (5, 70, 5, 13),     # planes of 4 n + 1 values
    (3, 66, 13, 10),    # 4 n + 2
    (23, 65, 9, 11),    # 4 n + 3: 575 units, two per thread of 1024
    (16, 2, 8, 16),     # 512 units: two per thread of 256
    (19, 72, 35, 35),   # eight units per thread, the last ones partly idle
    (8, 64, 64, 64),    # 8192 units: every thread full
    (8, 64, 64, 65),    # past them: reduce and map
    (4, 5, 64, 64),     # few channels: 4096 units
    (4, 5, 64, 66),     # past them
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("lead", [0, 1])
def test_training_step(module, dev, shape, lead):
    """Forward and backward, alone, with the ReLU behind, with a residual addition and with the
    input gradient's channel sums; tensors at their allocation's start and one float past it."""
    n, c, h, w = shape
    r = np.random.default_rng(n * c * h * w)
    x = (r.standard_normal(shape) * 1.3 + 0.4).astype(np.float32)
    g, more = (r.standard_normal(shape).astype(np.float32) for _ in range(2))
    gamma = r.uniform(0.5, 1.5, c).astype(np.float32)
    beta = r.uniform(-0.1, 0.1, c).astype(np.float32)
    rm = r.uniform(-0.5, 0.5, c).astype(np.float32)
    rv = r.uniform(0.5, 2.0, c).astype(np.float32)

    def device(a=None):
        flat = torch.full((x.size + lead,), float("nan"), device=dev)[lead:].view(shape)
        return flat if a is None else flat.copy_(torch.from_numpy(a))

    xd, gd, mored = device(x), device(g), device(more)
    vec = lambda: torch.full((c,), float("nan"), device=dev)  # noqa: E731
    wd, bd = to_dev(gamma, dev), to_dev(beta, dev)
    out = {}
    for kind in ("plain", "relu", "add"):
        rmd, rvd, mean, inv, y = to_dev(rm, dev), to_dev(rv, dev), vec(), vec(), device()
        args = (xd, wd, bd, rmd, rvd, mean, inv)
        if kind == "plain":
            module.batch_norm_forward_train(*args, y)
        elif kind == "relu":
            module.batch_norm_relu_forward_train(*args, y)
        else:
            module.batch_norm_add_forward_train(*args, mored, y)
        out[kind] = dict(y=host(y), mean=host(mean), inv=host(inv), rm=host(rmd), rv=host(rvd))
    check_batch_norm_forward(out["plain"], x, gamma, beta, rm, rv)
    for k in ("mean", "inv", "rm", "rv"):
        assert np.array_equal(out["plain"][k], out["relu"][k])
        assert np.array_equal(out["plain"][k], out["add"][k])
    assert np.array_equal(out["relu"]["y"], oracle.relu(out["plain"]["y"]))
    assert np.array_equal(out["add"]["y"], out["plain"]["y"] + more)

    mean, inv = out["plain"]["mean"], out["plain"]["inv"]
    md, id = to_dev(mean, dev), to_dev(inv, dev)
    relu_y = device(out["relu"]["y"])
    masked = oracle.relu_backward(g, out["plain"]["y"])
    for relu in (None, relu_y):
        incoming = g if relu is None else masked
        dx, dw, db, total = device(), vec(), vec(), vec()
        if relu is None:
            module.batch_norm_backward_train(gd, xd, wd, md, id, dx, dw, db)
        else:
            module.batch_norm_relu_backward_train(gd, relu, xd, wd, md, id, dx, dw, db)
        got = dict(dx=host(dx), dw=host(dw), db=host(db))
        check_batch_norm_backward(got, incoming, x, gamma, mean, inv)
        summed, dw2, db2 = device(), vec(), vec()
        module.conv_batch_norm_backward_train(gd, relu, xd, wd, md, id, summed, dw2, db2, total)
        for a, b in ((summed, "dx"), (dw2, "dw"), (db2, "db")):
            assert np.array_equal(host(a), got[b])
        wide = got["dx"].astype(np.float64)
        assert_within(host(total), wide.sum((0, 2, 3)),
                      1e-6 * np.abs(wide).sum((0, 2, 3)) + 1e-7, "input gradient sums")


@pytest.mark.parametrize("shape,by_slices", [
    ((32, 64, 32, 32), True),     # few channels with many whole units: every CU loads a share
    ((41, 79, 28, 28), True),
    ((32, 96, 32, 32), True),
    ((32, 64, 28, 24), False),    # up to six units per thread
    ((41, 96, 28, 28), False),
    ((32, 128, 32, 32), False),
    ((26, 64, 35, 35), False),    # no whole units
])
def test_forward_of_few_channels(dev, shape, by_slices):
    """The forward by slices leaves its partial sums in the workspace; the one by channels leaves
    the workspace as it was."""
    n, c, h, w = shape
    x = torch.randn(shape, device=dev)
    y = torch.empty_like(x)
    one = [torch.ones(c, device=dev) for _ in range(6)]
    size = ox.batch_norm_workspace_size(n, c, h * w)
    work = torch.full((size // 4,), float("nan"), device=dev)
    ox.check(ox.lib().oxh_batch_norm_forward_train(
        ox.current_stream(), n, c, h * w, 0.1, 1e-5, x.data_ptr(), *(t.data_ptr() for t in one),
        y.data_ptr(), work.data_ptr(), size))
    assert bool(work.isnan().all()) != by_slices
    ref = (x - x.mean((0, 2, 3), keepdim=True)) * (x.var((0, 2, 3), correction=0,
                                                         keepdim=True) + 1e-5).rsqrt() + 1
    assert float((y - ref).abs().max()) < 1e-4  # |x| < 7: some ulps of 2^-21


def test_values_that_are_not_finite(module, dev):
    """An infinity or a NaN takes its own channel alone with it, in the forward and (there in the
    incoming gradient) in the backward; the ReLU behind turns its NaN to 0."""
    shape = (19, 72, 35, 35)
    r = np.random.default_rng(3)
    x, g = (r.standard_normal(shape).astype(np.float32) for _ in range(2))
    gamma = r.uniform(0.5, 1.5, 72).astype(np.float32)
    beta, rm, rv = np.full(72, 0.1, np.float32), np.zeros(72, np.float32), np.ones(72, np.float32)

    def forward(values, relu):
        call = module.batch_norm_relu_forward_train if relu else module.batch_norm_forward_train
        out = [torch.empty(72, device=dev) for _ in range(2)] + [torch.empty(shape, device=dev)]
        call(to_dev(values, dev), to_dev(gamma, dev), to_dev(beta, dev), to_dev(rm, dev),
             to_dev(rv, dev), *out)
        return [host(t) for t in out]

    bad = x.copy()
    bad[3, 5, 2, 7], bad[4, 6, 0, 1] = np.inf, np.nan
    fine = np.delete(np.arange(72), [5, 6])
    for relu in (False, True):
        for a, b in zip(forward(x, relu), forward(bad, relu)):
            assert np.array_equal(*(t[fine] if t.ndim == 1 else t[:, fine] for t in (a, b)))
            if a.ndim > 1:
                assert (b[:, 5:7] == 0).all() if relu else np.isnan(b[:, 5:7]).all()
    ref = oracle.bn_forward(bad, gamma, beta, rm, rv, True, 0.1, 1e-5)[0]
    assert np.array_equal(np.isnan(ref), np.isnan(forward(bad, False)[2]))

    mean, inv, y = forward(x, True)
    g[2, 9, 1, 1], g[1, 10, 3, 3], y[2, 9, 1, 1], y[1, 10, 3, 3] = np.nan, -np.inf, 1.0, 1.0
    for relu in (False, True):
        dx, dw, db = torch.empty(shape, device=dev), *(torch.empty(72, device=dev) for _ in "wb")
        rest = (to_dev(x, dev), to_dev(gamma, dev), to_dev(mean, dev), to_dev(inv, dev), dx, dw, db)
        if relu:
            module.batch_norm_relu_backward_train(to_dev(g, dev), to_dev(y, dev), *rest)
        else:
            module.batch_norm_backward_train(to_dev(g, dev), *rest)
        incoming = oracle.relu_backward(g, y) if relu else g
        for got, want in zip((dx, dw, db), oracle.bn_backward(incoming, x, gamma, mean, inv, True)):
            got = host(got)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
            np.testing.assert_allclose(got[np.isfinite(want)], want[np.isfinite(want)], rtol=1e-3,
                                       atol=1e-3)
