"""The work that programs built on this package have it do, as timed cases.

Two kinds of programs use the package: those that call the eager operators
(`vkml_amd.ops`) on device arrays they own, with `out=` buffers they keep, and
those that build a network from `vkml_amd.nn` and replay its training step
(`vkml_amd.tensor.CapturedStep`). The cases cover both: matrix products in the
three layouts that a layer's forward and backward passes emit, from the smallest
layer to 4096 cubed, the K-dominant weight gradient, the matrix-vector product, a
convolution layer forward and backward, row softmax, reductions, and one training
step of a small fully connected and of a small convolutional network. Everything is
float32, the package's compute type.

Arrays are device memory of the package's own allocator; the outputs are returned
as torch tensors over the same memory (nothing is copied).
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from vkml_amd import nn, ops, optim
from vkml_amd import tensor as T
from vkml_amd.device import DeviceArray, backend


# ---- the cases ----------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # A small classifier's first layer on one batch, x @ W^T: launch latency.
        dict(name="linear_64x128x784", kind="matmul", layout="nt", batch=1, m=64, n=128, k=784),
        # An ordinary hidden layer's forward product, x @ W^T.
        dict(name="linear_1024", kind="matmul", layout="nt", batch=1, m=1024, n=1024, k=1024),
        # A plain product whose sizes fit no tile and no 16-byte row: user data.
        dict(name="matmul_ragged", kind="matmul", layout="nn", batch=1, m=1000, n=1501, k=777),
        # The largest product of the package's own sweep that is quoted, A @ B.
        dict(name="matmul_4096", kind="matmul", layout="nn", batch=1, m=4096, n=4096, k=4096),
        # A layer's weight gradient over a long batch, A^T @ B: few outputs, long K.
        dict(name="wgrad_128x784x16384", kind="matmul", layout="tn", batch=1, m=128, n=784, k=16384),
        # Single-sample inference through a square layer.
        dict(name="gemv_4096", kind="gemv", m=4096, k=4096),
        # A 3x3 layer's forward pass on 32x32 images.
        dict(name="conv_forward_32x32", kind="conv_forward", batch=128, cin=64, cout=128, hw=32, window=3, stride=1,
             pad=1),
        # The same layer behind a 2x2 pool: the gradients of its input and weights.
        dict(name="conv_backward_16x16", kind="conv_backward", batch=128, cin=64, cout=128, hw=16, window=3, stride=1,
             pad=1),
        # Class probabilities of a large batch.
        dict(name="softmax_4096x1000", kind="softmax", rows=4096, cols=1000, log=False),
        # Per-row statistics of an activation matrix: sum and maximum.
        dict(name="reduce_8192x4096", kind="reduce", rows=8192, cols=4096, axis=1),
        # One replayed training step of a 784-128-10 classifier, batch 64: latency.
        dict(name="mlp_step_64", kind="mlp_step", batch=64, hidden=128),
        # One replayed training step of the two-convolution network, batch 128.
        dict(name="cnn_step_128", kind="cnn_step", batch=128),
    ]


def _log_size(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    """One more case of the listed ranges: half of the sizes odd, the rest multiples of what layers use."""
    kind = rng.choice(["matmul"] * 5 + ["gemv"] + ["conv_forward", "conv_backward"] * 2
                      + ["softmax", "reduce", "mlp_step", "cnn_step"])

    def size(lo, hi, unit=16):
        v = _log_size(rng, lo, hi)
        return v if rng.random() < 0.5 else max(lo, v // unit * unit)

    if kind == "matmul":
        while True:
            c = dict(kind=kind, layout=rng.choice(["nn", "nt", "tn"]), batch=rng.choice([1, 1, 1, 4, 16]),
                     m=size(64, 4096), n=size(64, 4096), k=size(64, 16384))
            if c["batch"] * c["m"] * c["n"] * c["k"] <= 4096 ** 3 and c["batch"] * (
                    c["m"] * c["k"] + c["k"] * c["n"] + c["m"] * c["n"]) <= 1 << 27:
                return c
    if kind == "gemv":
        return dict(kind=kind, m=size(512, 8192), k=size(512, 8192))
    if kind in ("conv_forward", "conv_backward"):
        while True:
            window = rng.choice([1, 3, 3, 5])
            c = dict(kind=kind, batch=size(16, 128), cin=rng.choice([3, 16, 32, 64, 96, 128]),
                     cout=rng.choice([32, 64, 96, 128]), hw=rng.randint(7, 32), window=window,
                     stride=rng.choice([1, 1, 2]), pad=window // 2)
            if work(c)["flops"] <= 2 * 4096 ** 3:
                return c
    if kind == "softmax":
        cols = size(100, 32768)
        return dict(kind=kind, rows=max(16, min(16384, (1 << 25) // cols >> rng.randint(0, 4))), cols=cols,
                    log=rng.random() < 0.5)
    if kind == "reduce":
        return dict(kind=kind, rows=size(256, 8192), cols=size(256, 8192), axis=rng.randint(0, 1))
    if kind == "mlp_step":
        return dict(kind=kind, batch=size(16, 512), hidden=size(64, 1024))
    return dict(kind=kind, batch=size(8, 128))


# ---- device arrays and torch tensors over the same memory ---------------------

class _Span:
    """Device memory as torch.as_tensor takes it; holds the owner of the memory."""

    def __init__(self, owner, ptr: int, shape, strides, dtype):
        item = np.dtype(dtype).itemsize
        self.owner = owner
        self.__cuda_array_interface__ = {
            "data": (ptr, False), "shape": tuple(shape), "strides": tuple(s * item for s in strides),
            "typestr": np.dtype(dtype).str, "version": 2}


def _torch_of(a: DeviceArray) -> torch.Tensor:
    return torch.as_tensor(_Span(a.buffer, a.ptr, a.shape, a.strides, a.dtype), device="cuda")


def _torch_of_tensor(t: T.Tensor) -> torch.Tensor:
    n = t.node
    return torch.as_tensor(_Span(n.storage, n.storage.ptr + n.offset * n.itemsize, n.shape, n.strides, n.dtype),
                           device="cuda")


def _device(values: torch.Tensor) -> DeviceArray:
    """The package's own array holding `values`."""
    a = DeviceArray(tuple(values.shape), {torch.float32: np.float32, torch.int64: np.int64}[values.dtype])
    _torch_of(a).copy_(values)
    return a


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


# ---- inputs, from the seed alone ----------------------------------------------

def _window_count(case) -> int:
    return (case["hw"] + 2 * case["pad"] - case["window"]) // case["stride"] + 1


def _inputs(case, seed) -> dict[str, torch.Tensor]:
    g = _generator(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale

    def uniform(*shape, lo=-1.0, hi=1.0):
        return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo

    kind = case["kind"]
    if kind == "matmul":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        lead = (b,) if b > 1 else ()
        shape_a = lead + ((k, m) if case["layout"] == "tn" else (m, k))
        shape_b = lead + ((n, k) if case["layout"] == "nt" else (k, n))
        return {"a": normal(*shape_a), "b": normal(*shape_b)}
    if kind == "gemv":
        return {"a": normal(case["m"], case["k"]), "x": normal(case["k"])}
    if kind in ("conv_forward", "conv_backward"):
        out = _window_count(case)
        bound = 1.0 / math.sqrt(case["cin"] * case["window"] ** 2)
        d = {"x": uniform(case["batch"], case["cin"], case["hw"], case["hw"]),
             "w": uniform(case["cout"], case["cin"], case["window"], case["window"], lo=-bound, hi=bound)}
        if kind == "conv_backward":
            d["grad"] = normal(case["batch"], case["cout"], out, out)
        return d
    if kind == "softmax":
        return {"x": normal(case["rows"], case["cols"], scale=2.0)}
    if kind == "reduce":
        return {"x": normal(case["rows"], case["cols"])}
    if kind == "mlp_step":
        return {"x": uniform(case["batch"], 1, 28, 28, lo=0.0),
                "y": torch.randint(0, 10, (case["batch"],), generator=g, device="cuda")}
    return {"x": uniform(case["batch"], 3, 32, 32),
            "y": torch.randint(0, 100, (case["batch"],), generator=g, device="cuda")}


# ---- networks and their optimiser ---------------------------------------------

def _network(case, seed):
    """The network of a training case with its seeded Kaiming-uniform weights, and the learning rate."""
    nn.manual_seed(seed)
    if case["kind"] == "mlp_step":
        h = case["hidden"]
        return nn.Sequential(nn.Flatten(), nn.Linear(784, h), nn.ReLU(), nn.Linear(h, 10)), 0.1
    return nn.Sequential(nn.Conv2d(3, 64, 3, padding=1), nn.ReLU(), nn.MaxPool2d(2),
                         nn.Conv2d(64, 128, 3, padding=1), nn.ReLU(), nn.MaxPool2d(2), nn.Flatten(),
                         nn.Linear(8192, 256), nn.ReLU(), nn.Linear(256, 100)), 0.01


MOMENTUM = 0.9


# ---- prepare and run ----------------------------------------------------------

def prepare(case, seed):
    backend()
    kind = case["kind"]
    values = _inputs(case, seed)
    state = {"case": case, **{k: _device(v) for k, v in values.items()}}
    torch.cuda.synchronize()  # the package's stream does not wait for torch's
    if kind in ("mlp_step", "cnn_step"):
        model, lr = _network(case, seed)
        opt = optim.SGD(model.parameters(), lr=lr, momentum=MOMENTUM)

        def step(x, y):
            opt.zero_grad()
            loss = nn.cross_entropy(model(x), y)
            loss.backward()
            opt.step()
            return loss

        state["step"] = T.CapturedStep(step, values["x"].cpu().numpy(), values["y"].cpu().numpy())
        state["model"], state["opt"] = model, opt
        state["weights"] = [_torch_of_tensor(p) for p in model.parameters()]
        state["grads"] = [_torch_of_tensor(p.grad) for p in model.parameters()]
        return state
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        if case["layout"] == "tn":
            state["a"] = state["a"].transpose()
        if case["layout"] == "nt":
            state["b"] = state["b"].transpose()
        outs = [(*lead, case["m"], case["n"])]
    elif kind == "gemv":
        outs = [(case["m"],)]
    elif kind == "conv_forward":
        out = _window_count(case)
        outs = [(case["batch"], case["cout"], out, out)]
    elif kind == "conv_backward":
        outs = [(case["batch"], case["cin"], case["hw"], case["hw"]),
                (case["cout"], case["cin"] * case["window"] ** 2)]
    elif kind == "softmax":
        outs = [(case["rows"], case["cols"])]
    else:
        outs = [(case["rows"] if case["axis"] == 1 else case["cols"],)] * 2
    state["out"] = [DeviceArray(s) for s in outs]
    state["result"] = [_torch_of(o) for o in state["out"]]
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind in ("mlp_step", "cnn_step"):
        loss = state["step"](state["x"], state["y"])[0]
        return {"loss": loss, "weights": state["weights"], "grads": state["grads"]}
    out = state["out"]
    if kind == "matmul":
        ops.matmul(state["a"], state["b"], out=out[0])
    elif kind == "gemv":
        ops.gemv(state["a"], state["x"], out=out[0])
    elif kind == "conv_forward":
        ops.conv2d(state["x"], state["w"], case["stride"], case["pad"], out=out[0])
    elif kind == "conv_backward":
        ops.conv2d_input_grad(state["grad"], state["w"], (case["hw"], case["hw"]), case["stride"], case["pad"],
                              out=out[0])
        ops.conv2d_weight_grad_sum(state["x"], state["grad"], case["window"], case["stride"], case["pad"],
                                   out=out[1])
    elif kind == "softmax":
        ops.softmax(state["x"], -1, case["log"], out=out[0])
    else:
        ops.sum(state["x"], [case["axis"]], out=out[0])
        ops.amax(state["x"], [case["axis"]], out=out[1])
    return state["result"]


# ---- what a pass cannot do without ---------------------------------------------

def work(case) -> dict:
    kind = case["kind"]
    if kind == "matmul":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"bytes": 4 * b * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}
    if kind == "gemv":
        m, k = case["m"], case["k"]
        return {"bytes": 4 * (m * k + m + k), "flops": 2 * m * k}
    if kind in ("conv_forward", "conv_backward"):
        out = _window_count(case) ** 2
        ck = case["cin"] * case["window"] ** 2
        image, grad, weight = case["batch"] * case["cin"] * case["hw"] ** 2, case["batch"] * case["cout"] * out, \
            case["cout"] * ck
        product = 2 * case["batch"] * case["cout"] * out * ck
        if kind == "conv_forward":
            return {"bytes": 4 * (image + weight + grad), "flops": product}
        return {"bytes": 4 * (2 * image + 2 * weight + grad), "flops": 2 * product}
    if kind == "softmax":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 4 * case["rows"] * case["cols"]}
    if kind == "reduce":
        kept = case["rows"] if case["axis"] == 1 else case["cols"]
        return {"bytes": 4 * (case["rows"] * case["cols"] + 2 * kept), "flops": 2 * case["rows"] * case["cols"]}
    b = case["batch"]
    if kind == "mlp_step":
        h = case["hidden"]
        params = 784 * h + h + 10 * h + 10
        products = 2 * b * (2 * 784 * h + 3 * h * 10)
        image = 784
    else:
        params = 64 * 27 + 64 + 128 * 576 + 128 + 8192 * 256 + 256 + 256 * 100 + 100
        products = 2 * b * (2 * 1024 * 64 * 27 + 3 * 256 * 128 * 576 + 3 * 8192 * 256 + 3 * 256 * 100)
        image = 3 * 1024
    # a step reads and writes the weights and their velocities and leaves the gradients
    return {"bytes": 4 * (5 * params + b * image) + 8 * b, "flops": products}


def tolerance(case):
    kind = case["kind"]
    if kind in ("mlp_step", "cnn_step"):
        # a near tie in a pool window or at a relu's zero moves one gradient
        # value; without one the gradients agree to 2e-6
        return {"rel": 1e-4, "max": 1e-2}
    if kind == "softmax":
        return {"rel": 1e-6, "max": 1e-5}
    if kind in ("gemv", "reduce"):
        return {"rel": 1e-6, "max": 2e-5}
    # 32-bit sums of up to 16384 (products) or 131072 (batch-folded) terms:
    # 1.1e-6 from the 64-bit result at K = 4096 in one chain
    return {"rel": 5e-6, "max": 1e-4}


# ---- the same in 64 bits, without this package ----------------------------------

def _columns(x, case):
    return F.unfold(x, case["window"], padding=case["pad"], stride=case["stride"])


def _conv64(x, w, pad):
    n, _, h, wd = x.shape
    k = w.shape[-1]
    cols = F.unfold(x, k, padding=pad)
    return (w.reshape(w.shape[0], -1) @ cols).reshape(n, w.shape[0], h + 2 * pad - k + 1, wd + 2 * pad - k + 1)


def _weights64(case, seed):
    """The seeded weights in the network's order: each layer's weight, uniform in +-1/sqrt(fan in), then its bias."""
    rng = np.random.default_rng(seed)
    shapes = [(case["hidden"], 784), (10, case["hidden"])] if case["kind"] == "mlp_step" else \
        [(64, 3, 3, 3), (128, 64, 3, 3), (256, 8192), (100, 256)]
    out = []
    for s in shapes:
        bound = 1.0 / math.sqrt(math.prod(s[1:]))
        for shape in (s, s[:1]):
            w = rng.uniform(-bound, bound, size=shape).astype(np.float32)
            out.append(torch.from_numpy(w).double().cuda().requires_grad_(True))
    return out


def _step64(case, p, x, y):
    if case["kind"] == "mlp_step":
        h = torch.relu(x.reshape(len(x), -1) @ p[0].T + p[1])
        return F.cross_entropy(h @ p[2].T + p[3], y)
    h = F.max_pool2d(torch.relu(_conv64(x, p[0], 1) + p[1].reshape(-1, 1, 1)), 2)
    h = F.max_pool2d(torch.relu(_conv64(h, p[2], 1) + p[3].reshape(-1, 1, 1)), 2)
    h = torch.relu(h.reshape(len(x), -1) @ p[4].T + p[5])
    return F.cross_entropy(h @ p[6].T + p[7], y)


def exact(case, seed):
    kind = case["kind"]
    v = {k: t.double() if t.is_floating_point() else t for k, t in _inputs(case, seed).items()}
    if kind == "matmul":
        a = v["a"].mT if case["layout"] == "tn" else v["a"]
        b = v["b"].mT if case["layout"] == "nt" else v["b"]
        return [torch.matmul(a, b)]
    if kind == "gemv":
        return [v["a"] @ v["x"]]
    if kind in ("conv_forward", "conv_backward"):
        flat, cols = v["w"].reshape(case["cout"], -1), _columns(v["x"], case)
        out = _window_count(case)
        if kind == "conv_forward":
            return [(flat @ cols).reshape(case["batch"], case["cout"], out, out)]
        grad = v["grad"].reshape(case["batch"], case["cout"], -1)
        dx = F.fold(flat.T @ grad, (case["hw"], case["hw"]), case["window"], padding=case["pad"],
                    stride=case["stride"])
        dw = grad.transpose(0, 1).reshape(case["cout"], -1) @ cols.transpose(1, 2).reshape(-1, cols.shape[1])
        return [dx, dw]
    if kind == "softmax":
        return [torch.log_softmax(v["x"], -1) if case["log"] else torch.softmax(v["x"], -1)]
    if kind == "reduce":
        return [v["x"].sum(case["axis"]), v["x"].amax(case["axis"])]
    # training: prepare() has made the first step, run() makes the second
    p, velocity = _weights64(case, seed), None
    lr = 0.1 if kind == "mlp_step" else 0.01
    for _ in range(2):
        loss = _step64(case, p, v["x"], v["y"])
        grads = torch.autograd.grad(loss, p)
        velocity = list(grads) if velocity is None else [MOMENTUM * u + g for u, g in zip(velocity, grads)]
        p = [(w - lr * u).detach().requires_grad_(True) for w, u in zip(p, velocity)]
    return {"loss": loss.detach(), "weights": [w.detach() for w in p], "grads": list(grads)}
