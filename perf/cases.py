"""The workloads this framework's speed is measured on: the calls a training or inference program
makes through the public entry points, at sizes from the smallest call to the largest.

A case is a dict of plain values; ``kind`` says which path it takes:

* ``train``: one training step of MobileNetV4-Conv-S (forward, cross entropy, backward, AdamW)
  replayed from its graph, as ``training.TrainingStep`` runs it, some way into a training run
  (the optimizer's moments are those of earlier steps);
* ``eval``: its inference forward from the running statistics (``training.EvalForward``);
* ``conv``: one convolution layer, forward and backward (input, weight and bias gradients);
* ``batch_norm``: one BatchNorm2d layer (``relu``: with the ReLU behind it), training forward
  and backward;
* ``cross_entropy``: loss and logit gradient over a batch of rows;
* ``adamw``: one optimizer step over a flat parameter vector, in place;
* ``plan``: one replay of the compiled plan of relu((a + b) * c).

All data is float32, the one type the framework computes in.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch
import torch.nn.functional as F

_PACKAGE = Path(__file__).resolve().parents[1] / "oxide-beta_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

import jit  # noqa: E402
import oxide_hip as ox  # noqa: E402
import training  # noqa: E402

MOMENTUM, EPSILON = 0.1, 1e-5
LR, DECAY, BETA1, BETA2, ADAM_EPSILON, ADAM_STEP = 1e-3, 0.01, 0.9, 0.999, 1e-8, 10
TRAIN_LR, TRAIN_DECAY, TRAIN_STEP = 1e-3, 1e-4, 1000


def listed() -> list[dict]:
    return [
        # the MNIST example's training step at its batch size
        {"name": "train 28x28 b128", "kind": "train", "batch": 128, "classes": 10,
         "channels": 1, "resolution": 28},
        # the same network's 224 x 224 RGB variant with 1000 classes
        {"name": "train 224x224 b32", "kind": "train", "batch": 32, "classes": 1000,
         "channels": 3, "resolution": 224},
        # classifying one digit as it comes in: latency
        {"name": "eval 28x28 b1", "kind": "eval", "batch": 1, "classes": 10, "channels": 1,
         "resolution": 28},
        # classifying a batch of photographs
        {"name": "eval 224x224 b64", "kind": "eval", "batch": 64, "classes": 1000,
         "channels": 3, "resolution": 224},
        # a 1 x 1 expansion of an inverted bottleneck, outside the network
        {"name": "conv 1x1 64-192 56x56", "kind": "conv", "batch": 64, "in": 64, "out": 192,
         "height": 56, "width": 56, "kernel": 1, "stride": 1, "groups": 1},
        # a residual network's 3 x 3 layer
        {"name": "conv 3x3 64-64 56x56", "kind": "conv", "batch": 32, "in": 64, "out": 64,
         "height": 56, "width": 56, "kernel": 3, "stride": 1, "groups": 1},
        # the BatchNorm2d layer of the benchmark
        {"name": "bn 128c 56x56", "kind": "batch_norm", "batch": 64, "channels": 128,
         "height": 56, "width": 56, "relu": False},
        # BatchNorm2d and ReLU over odd planes (an odd input size), a ragged batch
        {"name": "bn relu 72c 35x35", "kind": "batch_norm", "batch": 19, "channels": 72,
         "height": 35, "width": 35, "relu": True},
        # the benchmark's cross entropy: a language model's vocabulary
        {"name": "ce 8192x32768", "kind": "cross_entropy", "batch": 8192, "classes": 32768},
        # an image classifier's loss, rows that are no multiple of anything
        {"name": "ce 509x1003", "kind": "cross_entropy", "batch": 509, "classes": 1003},
        # the benchmark's optimizer step
        {"name": "adamw 64Mi", "kind": "adamw", "elements": 1 << 26},
        # the benchmark's compiled plan
        {"name": "plan 4096x4096", "kind": "plan", "rows": 4096, "columns": 4096},
    ]


def _log(rng, low, high) -> int:
    """A whole number, uniform over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng) -> dict:
    kind = rng.choice(["train", "eval", "conv1", "convk", "depthwise", "batch_norm",
                       "cross_entropy", "adamw", "plan"])
    if kind in ("train", "eval"):
        channels, classes = rng.choice([(1, 10), (3, 1000), (3, rng.randint(2, 400))])
        resolution = rng.choice([28, 32, 64, 96, 128, 160, 192, 224])
        most = 32 if kind == "train" else 64
        batch = _log(rng, 16 if kind == "train" else 1,
                     min(256, most * 224 * 224 // resolution ** 2))
        return {"kind": kind, "batch": batch, "classes": classes, "channels": channels,
                "resolution": resolution}
    if kind in ("conv1", "convk", "depthwise"):
        k = 1 if kind == "conv1" else rng.choice([3, 3, 5])
        cin = _log(rng, 3 if kind == "convk" else 16, 128 if kind == "convk" else 960)
        cout = cin if kind == "depthwise" else _log(rng, 16, 128 if kind == "convk" else 960)
        if rng.random() < 0.6:  # most layers have channel counts of whole vectors
            cin = -(-cin // 8) * 8
            cout = cin if kind == "depthwise" else -(-cout // 8) * 8
        groups = cin if kind == "depthwise" else 1
        height = _log(rng, 4, 112)
        width = height if rng.random() < 0.7 else _log(rng, 4, 112)
        stride = 1 if kind == "conv1" else rng.choice([1, 2])
        # within the listed layers' tensors and products
        values = 64 * 192 * 56 * 56 / (max(cin, cout) * height * width)
        products = 32 * 64 * 64 * 9 * 56 * 56 / (cin * cout / groups * k * k * height * width)
        batch = _log(rng, 1, max(1, int(min(128, values, products))))
        return {"kind": "conv", "batch": batch, "in": cin, "out": cout, "height": height,
                "width": width, "kernel": k, "stride": stride, "groups": groups}
    if kind == "batch_norm":
        channels, height = _log(rng, 8, 960), _log(rng, 1, 112)
        width = height if rng.random() < 0.7 else _log(rng, 1, 112)
        most = 64 * 128 * 56 * 56 // (channels * height * width)
        return {"kind": kind, "batch": _log(rng, 2, max(2, min(256, most))),
                "channels": channels, "height": height, "width": width,
                "relu": rng.random() < 0.5}
    if kind == "cross_entropy":
        classes = _log(rng, 2, 100000)
        return {"kind": kind, "batch": _log(rng, 1, min(8192, (1 << 28) // classes)),
                "classes": classes}
    if kind == "adamw":
        return {"kind": kind, "elements": _log(rng, 1000, 1 << 26)}
    return {"kind": "plan", "rows": _log(rng, 1, 4096), "columns": _log(rng, 16, 4096)}


# ----------------------------------------------------------------------------- inputs

def _generator(case: dict, seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(0x6F786964 + 1000003 * int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _uniform(g, low, high, *shape):
    return torch.rand(shape, generator=g, device="cuda") * (high - low) + low


def _classes(g, n, classes):
    return torch.randint(0, classes, (n,), generator=g, device="cuda").float()


# The network, layer by layer: (in, out, kernel, stride, depthwise, relu); a block is a list of
# layers and whether its input is added to its output.
_UIB = [(64, 96, 192, 5, 5, 2), (96, 96, 192, 0, 3, 1), (96, 96, 192, 0, 3, 1),
        (96, 96, 192, 0, 3, 1), (96, 96, 192, 0, 3, 1), (96, 96, 384, 3, 0, 1),
        (96, 128, 576, 3, 3, 2), (128, 128, 512, 5, 5, 1), (128, 128, 512, 0, 5, 1),
        (128, 128, 384, 0, 5, 1), (128, 128, 512, 0, 3, 1), (128, 128, 512, 0, 3, 1)]


def _blocks(case: dict) -> list:
    blocks = [([(case["channels"], 32, 3, 2, False, True)], False),
              ([(32, 32, 3, 2, False, True), (32, 32, 1, 1, False, False)], False),
              ([(32, 96, 3, 2, False, True), (96, 64, 1, 1, False, False)], False)]
    for cin, cout, wide, start, middle, stride in _UIB:
        layers = [(cin, cin, start, 1, True, True)] if start else []
        layers.append((cin, wide, 1, 1, False, True))
        if middle:
            layers.append((wide, wide, middle, stride, True, True))
        layers.append((wide, cout, 1, 1, False, False))
        blocks.append((layers, stride == 1 and cin == cout))
    blocks.append(([(128, 960, 1, 1, False, True)], False))
    blocks.append("pool")
    blocks.append(([(960, 1280, 1, 1, False, True)], False))
    return blocks


def _layers(case: dict):
    """(layer, input size) of every ConvNormAct in order."""
    size = case["resolution"]
    for block in _blocks(case):
        if block == "pool":
            size = 1
            continue
        for layer in block[0]:
            yield layer, size
            size = (size + 2 * (layer[2] // 2) - layer[2]) // layer[3] + 1


def _network_inputs(case: dict, seed: int) -> dict:
    """Parameters in the model's order (per layer: weight, bias, gamma, beta; the classifier's
    weight and bias last), running statistics, images and labels."""
    g = _generator(case, seed)
    parameters, running = [], []
    for (cin, cout, k, _, depthwise, _), _ in _layers(case):
        fan = k * k * (1 if depthwise else cin)
        bound = math.sqrt(6.0 / fan)
        parameters += [_uniform(g, -bound, bound, cout, 1 if depthwise else cin, k, k),
                       _uniform(g, -0.05, 0.05, cout), _uniform(g, 0.5, 1.5, cout),
                       _uniform(g, -0.1, 0.1, cout)]
        running += [(0.1 * _normal(g, cout), _uniform(g, 0.5, 1.5, cout))]
    bound = math.sqrt(3.0 / 1280)
    parameters += [_uniform(g, -bound, bound, case["classes"], 1280, 1, 1),
                   _uniform(g, -0.05, 0.05, case["classes"])]
    # an earlier step's moments, of a scale that falls with depth as the gradients' does
    moments = []
    for i, p in enumerate(parameters if case["kind"] == "train" else []):
        scale = 0.003 ** (i / len(parameters))
        moments += [(_normal(g, *p.shape) * (0.3 * scale),
                     _uniform(g, 0.5, 1.5, *p.shape) * scale ** 2)]
    r = case["resolution"]
    shape = (case["batch"], case["channels"], r, r)
    if case["channels"] == 1:  # pixels k / 255
        images = torch.randint(0, 256, shape, generator=g, device="cuda").float() / 255.0
    else:  # normalized channels
        images = _normal(g, *shape)
    return {"parameters": parameters, "moments": moments, "running": running, "images": images,
            "labels": _classes(g, case["batch"], case["classes"])}


class _Buffer:
    """A device buffer that ``owner`` (a step, a model, a plan) frees, as torch takes it in: the
    tensor holds this object, and so its owner, for as long as it lives."""

    def __init__(self, pointer: int, shape, dtype, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(pointer), False),
                                         "typestr": np.dtype(dtype).str, "shape": tuple(shape),
                                         "strides": None, "version": 2}


def _tensor(pointer: int, shape, dtype, owner) -> torch.Tensor:
    return torch.as_tensor(_Buffer(pointer, shape, dtype, owner), device="cuda")


def _view(v, owner) -> torch.Tensor:
    return _tensor(v.ptr, v.shape, v.dtype, owner)


_kernels = None


def _module() -> ox.LoadedModule:
    """The launchers, loaded once as a program loads them."""
    global _kernels
    if _kernels is None:
        _kernels = ox.load_kernels(0)
    return _kernels


def _conv_shape(case: dict):
    return ox.conv2d_shape(case["batch"], case["in"], case["height"], case["width"],
                           case["out"], case["kernel"], case["stride"], case["kernel"] // 2,
                           case["groups"])


def _conv_output(case: dict) -> tuple:
    pad, k, s = case["kernel"] // 2, case["kernel"], case["stride"]
    return (case["batch"], case["out"], (case["height"] + 2 * pad - k) // s + 1,
            (case["width"] + 2 * pad - k) // s + 1)


def _conv_inputs(case: dict, seed: int) -> tuple:
    """x (after a ReLU), weight, bias and the output's gradient."""
    g = _generator(case, seed)
    x = _normal(g, case["batch"], case["in"], case["height"], case["width"]).relu_()
    per_group = case["in"] // case["groups"]
    bound = math.sqrt(6.0 / (per_group * case["kernel"] ** 2))
    weight = _uniform(g, -bound, bound, case["out"], per_group, case["kernel"], case["kernel"])
    return x, weight, _uniform(g, -0.05, 0.05, case["out"]), _normal(g, *_conv_output(case))


def _bn_inputs(case: dict, seed: int) -> tuple:
    g = _generator(case, seed)
    c = case["channels"]
    shape = (case["batch"], c, case["height"], case["width"])
    return (_normal(g, *shape), _uniform(g, 0.5, 1.5, c), _uniform(g, -0.1, 0.1, c),
            _normal(g, *shape))


def _ce_inputs(case: dict, seed: int) -> tuple:
    g = _generator(case, seed)
    logits = _normal(g, case["batch"], case["classes"]).mul_(2.0)
    return logits, _classes(g, case["batch"], case["classes"])


def _adamw_inputs(case: dict, seed: int) -> tuple:
    """Parameters, gradients and the moments an earlier step's gradients left."""
    g = _generator(case, seed)
    n = case["elements"]
    p, grad, before = (_normal(g, n).mul_(s) for s in (0.02, 1e-3, 1e-3))
    return p, grad, before * 0.1, before * before * 0.001


def _plan_inputs(case: dict, seed: int) -> tuple:
    g = _generator(case, seed)
    return tuple(_uniform(g, -1.0, 1.0, case["rows"], case["columns"]) for _ in range(3))


# ----------------------------------------------------------------------------- state and pass

def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("train", "eval"):
        given = _network_inputs(case, seed)
        model = training.MobileNetV4ConvSmall(case["classes"], case["channels"],
                                              case["resolution"])
        for p, values in zip(model.parameters(), given["parameters"], strict=True):
            _view(p.value, model).copy_(values)
        if kind == "eval":
            for b, (mean, variance) in zip(model.batch_norms(), given["running"], strict=True):
                _view(b.device_running_mean, model).copy_(mean)
                _view(b.device_running_variance, model).copy_(variance)
            model.eval()
            step = training.EvalForward(model, case["batch"])
            outputs = {"logits": _view(step.logits, step)}
        else:
            step = training.TrainingStep(model, case["batch"], TRAIN_LR, TRAIN_DECAY)
            _view(step.targets, step).copy_(given["labels"])
            adamw = next(op.attrs for op in step.ops if op.kind == "adamw")
            by_parameter = {p.ptr: rest for p, *rest in adamw["tensors"]}
            parameters = [p.value for p in model.parameters()]
            for p, (first, second) in zip(parameters, given["moments"], strict=True):
                _view(by_parameter[p.ptr][1].view(p.shape), step).copy_(first)
                _view(by_parameter[p.ptr][2].view(p.shape), step).copy_(second)
            _view(adamw["step_counter"], step).fill_(TRAIN_STEP - 1)
            classifier = parameters[-2]
            gradient = by_parameter[classifier.ptr][0].view(classifier.shape)
            outputs = {"loss": _view(step.loss, step), "logits": _view(step.logits, step),
                       "classifier_gradient": _view(gradient, step),
                       "weights": [_view(p, step) for p in parameters if len(p.shape) == 4]}
        _view(step.input, step).copy_(given["images"])
        torch.cuda.synchronize()
        step.capture()
        return {"kind": kind, "step": step, "model": model, "outputs": outputs}
    if kind == "conv":
        x, weight, bias, gradient = _conv_inputs(case, seed)
        outputs = {"y": torch.empty_like(gradient), "dx": torch.empty_like(x),
                   "dweight": torch.empty_like(weight), "dbias": torch.empty_like(bias)}
        return {"kind": kind, "shape": _conv_shape(case), "inputs": (x, weight, bias, gradient),
                "outputs": outputs}
    if kind == "batch_norm":
        inputs = _bn_inputs(case, seed)
        c = case["channels"]
        vector = lambda value: torch.full((c,), value, device="cuda")  # noqa: E731
        outputs = {"y": torch.empty_like(inputs[0]), "dx": torch.empty_like(inputs[0]),
                   "mean": vector(0.0), "inverse_std": vector(0.0), "dweight": vector(0.0),
                   "dbias": vector(0.0), "running_mean": vector(0.0),
                   "running_variance": vector(1.0)}
        return {"kind": kind, "inputs": inputs, "relu": case["relu"], "outputs": outputs}
    if kind == "cross_entropy":
        logits, targets = _ce_inputs(case, seed)
        return {"kind": kind, "inputs": (logits, targets, torch.ones(1, device="cuda")),
                "outputs": {"loss": torch.empty(1, device="cuda"),
                            "gradient": torch.empty_like(logits)}}
    if kind == "adamw":
        p, gradient, m, v = _adamw_inputs(case, seed)
        return {"kind": kind, "gradient": gradient,
                "corrections": ox.adamw_corrections(BETA1, BETA2, ADAM_STEP),
                "outputs": {"parameter": p, "first_moment": m, "second_moment": v}}
    shape = (case["rows"], case["columns"])
    example = np.broadcast_to(np.float32(0), shape)  # a trace reads its shape alone
    traced = jit.trace([example] * 3, lambda v: ((v[0] + v[1]) * v[2]).relu())
    plan = traced.plan_for((shape,) * 3)
    for slot, values in zip(plan.plan.inputs, _plan_inputs(case, seed)):
        _tensor(plan.buffer(slot)[0], shape, np.float32, plan).copy_(values)
    torch.cuda.synchronize()
    return {"kind": kind, "plan": plan,
            "outputs": _tensor(plan.buffer(plan.plan.output)[0], shape, np.float32, plan)}


def run(state: dict):
    kind, out = state["kind"], state["outputs"]
    if kind in ("train", "eval"):
        state["step"].replay()
    elif kind == "conv":
        m, shape = _module(), state["shape"]
        x, weight, bias, gradient = state["inputs"]
        m.conv2d_forward(shape, x, weight, bias, out["y"])
        m.conv2d_backward(shape, gradient, x, weight, out["dx"], out["dweight"], out["dbias"])
    elif kind == "batch_norm":
        m = _module()
        x, weight, bias, gradient = state["inputs"]
        forward = (x, weight, bias, out["running_mean"], out["running_variance"], out["mean"],
                   out["inverse_std"], out["y"], MOMENTUM, EPSILON)
        backward = (x, weight, out["mean"], out["inverse_std"], out["dx"], out["dweight"],
                    out["dbias"])
        if state["relu"]:
            m.batch_norm_relu_forward_train(*forward)
            m.batch_norm_relu_backward_train(gradient, out["y"], *backward)
        else:
            m.batch_norm_forward_train(*forward)
            m.batch_norm_backward_train(gradient, *backward)
    elif kind == "cross_entropy":
        logits, targets, outer = state["inputs"]
        _module().cross_entropy_forward_backward(logits.shape[0], logits.shape[1], logits,
                                                 targets, outer, out["loss"], out["gradient"])
    elif kind == "adamw":
        p, m, v = out["parameter"], out["first_moment"], out["second_moment"]
        _module().adamw(LR, DECAY, BETA1, BETA2, *state["corrections"], ADAM_EPSILON, p,
                        state["gradient"], m, v, p, m, v)
    else:
        state["plan"].replay()
    return out


# ----------------------------------------------------------------------------- what it takes

def work(case: dict) -> dict:
    """Inputs read once and outputs written once; for a training step also the parameters,
    their gradients and moments, and every convolution's output, written by the forward and
    read by the backward."""
    kind = case["kind"]
    if kind in ("train", "eval"):
        values = products = kept = 0
        for (cin, cout, k, stride, depthwise, _), size in _layers(case):
            fan = k * k * (1 if depthwise else cin)
            out = (size + 2 * (k // 2) - k) // stride + 1
            values += cout * (fan + 3)
            products += cout * fan * out * out * case["batch"]
            kept += cout * out * out * case["batch"]
        values += case["classes"] * 1281
        products += case["classes"] * 1280 * case["batch"]
        images = case["batch"] * case["channels"] * case["resolution"] ** 2
        logits = case["batch"] * case["classes"]
        if kind == "eval":
            return {"bytes": 4 * (images + values + logits), "flops": 2 * products}
        return {"bytes": 4 * (images + 7 * values + 2 * kept + 2 * logits),
                "flops": 6 * products}
    if kind == "conv":
        n, cout, oh, ow = _conv_output(case)
        fan = case["in"] // case["groups"] * case["kernel"] ** 2
        x, y = n * case["in"] * case["height"] * case["width"], n * cout * oh * ow
        return {"bytes": 4 * (2 * x + 2 * y + 2 * cout * fan), "flops": 6 * y * fan}
    if kind == "batch_norm":
        n = case["batch"] * case["channels"] * case["height"] * case["width"]
        return {"bytes": 16 * n, "flops": 14 * n}
    if kind == "cross_entropy":
        n = case["batch"] * case["classes"]
        return {"bytes": 8 * n, "flops": 8 * n}
    if kind == "adamw":
        return {"bytes": 28 * case["elements"], "flops": 15 * case["elements"]}
    n = case["rows"] * case["columns"]
    return {"bytes": 16 * n, "flops": 3 * n}


def tolerance(case: dict):
    """Elementwise results keep their bits; sums in another order differ by their rounding.  A
    ReLU whose input another rounding moves past zero lets a whole gradient through, or none, and
    a network carries that through the layers before it into the weights and, over the next
    step, the logits (up to 0.3 % between 32 and 64 bits)."""
    if case["kind"] in ("plan", "adamw"):
        return "exact"
    if case["kind"] == "train":
        return {"rel": 1e-2}
    if case["kind"] == "batch_norm" and case["relu"]:
        return {"rel": 1e-3, "max": 0.99}
    return {"rel": 1e-5}


# ----------------------------------------------------------------------------- in 64 bits

def _exact_network(case: dict, seed: int) -> dict:
    """The updated weights have no such value: they hang on which ReLU inputs a rounding moves
    past zero.  Nothing that the loss, the logits and the classifier's gradient hang on does."""
    given = _network_inputs(case, seed)
    train = case["kind"] == "train"
    parameters = [p.double() for p in given["parameters"]]
    running = [(m.double(), v.double()) for m, v in given["running"]]
    x, layer_at = given["images"].double(), 0
    for block in _blocks(case):
        if block == "pool":
            x = x.mean((2, 3), keepdim=True)
            continue
        layers, residual = block
        before = x
        for cin, _, k, stride, depthwise, relu in layers:
            weight, bias, gamma, beta = parameters[4 * layer_at:4 * layer_at + 4]
            x = F.conv2d(x, weight, bias, stride, k // 2, 1, cin if depthwise else 1)
            mean, variance = running[layer_at]
            x = F.batch_norm(x, mean, variance, gamma, beta, train, MOMENTUM, EPSILON)
            x = x.relu() if relu else x
            layer_at += 1
        x = x + before if residual else x
    logits = F.conv2d(x, *parameters[-2:]).flatten(1)
    if not train:
        return {"logits": logits}
    labels = given["labels"].long()
    error = (logits.softmax(1) - F.one_hot(labels, case["classes"])) / case["batch"]
    return {"loss": F.cross_entropy(logits, labels).reshape(1), "logits": logits,
            "classifier_gradient": (error.t() @ x.flatten(1)).reshape(parameters[-2].shape),
            "weights": [None] * sum(p.dim() == 4 for p in parameters)}


def exact(case: dict, seed: int):
    kind = case["kind"]
    with torch.backends.cudnn.flags(enabled=False):
        if kind in ("train", "eval"):
            return _exact_network(case, seed)
        if kind == "conv":
            x, weight, bias, gradient = (t.double() for t in _conv_inputs(case, seed))
            leaves = [t.requires_grad_(True) for t in (x, weight, bias)]
            y = F.conv2d(x, weight, bias, case["stride"], case["kernel"] // 2, 1,
                         case["groups"])
            dx, dweight, dbias = torch.autograd.grad(y, leaves, gradient)
            return {"y": y.detach(), "dx": dx, "dweight": dweight, "dbias": dbias}
    if kind == "batch_norm":
        x, weight, bias, gradient = (t.double() for t in _bn_inputs(case, seed))
        c = lambda v: v.reshape(1, -1, 1, 1)  # noqa: E731
        count = x.numel() // x.shape[1]
        mean = x.mean((0, 2, 3))
        variance = (x - c(mean)).square().mean((0, 2, 3))
        inverse_std = (variance + EPSILON).rsqrt()
        xhat = (x - c(mean)) * c(inverse_std)
        y = xhat * c(weight) + c(bias)
        if case["relu"]:
            gradient = gradient * (y > 0)
            y = y.relu()
        dweight, dbias = (gradient * xhat).sum((0, 2, 3)), gradient.sum((0, 2, 3))
        dx = c(weight * inverse_std) * (gradient - c(dbias / count) - xhat * c(dweight / count))
        if case["relu"]:  # at a y that rounds to zero or past it, they have no one value
            dx = dweight = dbias = None
        return {"y": y, "dx": dx, "mean": mean, "inverse_std": inverse_std, "dweight": dweight,
                "dbias": dbias, "running_mean": MOMENTUM * mean,
                "running_variance": 1.0 - MOMENTUM + MOMENTUM * variance * count / (count - 1)}
    if kind == "cross_entropy":
        logits, targets = _ce_inputs(case, seed)
        log_p = logits.double().log_softmax(1)
        at = targets.long().unsqueeze(1)
        loss = -log_p.gather(1, at).mean().reshape(1)
        gradient = log_p.exp_().scatter_add_(1, at, torch.full_like(at, -1, dtype=torch.double))
        return {"loss": loss, "gradient": gradient.div_(case["batch"])}
    if kind == "adamw":
        p, gradient, m, v = (t.double() for t in _adamw_inputs(case, seed))
        m = BETA1 * m + (1 - BETA1) * gradient
        v = BETA2 * v + (1 - BETA2) * gradient.square()
        update = (m / (1 - BETA1 ** ADAM_STEP)) / ((v / (1 - BETA2 ** ADAM_STEP)).sqrt()
                                                   + ADAM_EPSILON)
        return {"parameter": p * (1 - LR * DECAY) - LR * update, "first_moment": m,
                "second_moment": v}
    a, b, c = (t.double() for t in _plan_inputs(case, seed))
    return ((a + b) * c).relu()
