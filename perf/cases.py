"""What is timed: the calls that a program on this package makes, over the range of sizes it makes them with.

Most cases keep their operands on the device (``device_tensor``), as a training loop does, and leave
results and gradients there; they are handed back as torch tensors over the same memory.  The two
``net`` cases take host arrays in and read every result on the host, which is how a program written
for NumPy arrays uses the package.
"""

import math

import numpy as np
import torch

import mygrad_amd as mg
from mygrad_amd.nnet import batchnorm, conv_nd, max_pool, relu

_TORCH = {"f32": torch.float32, "f64": torch.float64}
_NUMPY = {"f32": np.float32, "f64": np.float64}
_BYTES = {"f32": 4, "f64": 8}
_AXES = "0", "1", "2"  # suffixes of the per-axis entries of a case


# ----------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest layer in use: a first layer on 32 x 32 images in the reference's default dtype, where
        # launches and the host side of a step count
        _conv("conv-small-f64", "f64", 32, 3, 16, (32, 32), (3, 3), (1, 1), (1, 1), (1, 1)),
        # the 3x3 layer of a residual network's first stage: the bulk of a convolutional network's time
        _conv("conv3x3-f32", "f32", 128, 64, 64, (56, 56), (3, 3), (1, 1), (1, 1), (1, 1)),
        # the layer between two stages: halves the rows, doubles the channels; odd extents
        _conv("conv-strided-f32", "f32", 128, 128, 256, (27, 27), (3, 3), (2, 2), (1, 1), (1, 1)),
        # a wide receptive field in double precision: stride along one axis only, dilated, padded
        _conv("conv-dilated-f64", "f64", 16, 32, 32, (127, 128), (5, 5), (2, 1), (4, 4), (2, 2)),
        # a layer over long sequences, with channel counts and a length that fit no tile
        _conv("conv1d-ragged-f32", "f32", 16, 45, 83, (16001,), (9,), (1,), (4,), (1,)),
        # volumes: convolution, pooling and a loss as one graph
        {"name": "chain3d-f32", "kind": "chain", "dtype": "f32", "n": 8, "c": 16, "f": 32, "nd": 3, "x0": 32, "x1": 64, "x2": 64},
        # overlapping windows in double precision, no convolution around them
        {"name": "pool-overlap-f64", "kind": "pool", "dtype": "f64", "n": 64, "c": 64, "nd": 2, "g": 27, "window": 3, "stride": 2},
        # the first block of an image network: 7x7 filters on constant images, batchnorm, relu, pooling
        {"name": "stem-f32", "kind": "stem", "dtype": "f32", "n": 64, "f": 64, "p": 56},
        # one training step of a small image classifier on host arrays, every gradient read
        {"name": "net-train-f32", "kind": "train", "dtype": "f32", "n": 100, "side": 32, "c": 3, "f1": 16, "f2": 32, "window": 3, "classes": 10},
        # the same network answering a few images: latency
        {"name": "net-infer-f32", "kind": "infer", "dtype": "f32", "n": 8, "side": 32, "c": 3, "f1": 16, "f2": 32, "window": 3, "classes": 10},
        # a wide dense layer: the largest products
        {"name": "dense-f32", "kind": "dense", "dtype": "f32", "m": 4096, "k": 4096, "n": 4096},
        # two stacks of small matrices of uneven extents, as between the heads of an attention layer
        {"name": "stacks-f32", "kind": "stacks", "dtype": "f32", "b": 96, "m": 197, "k": 64, "n": 197},
    ]


def draw(rng):
    kind = rng.choice(("conv",) * 6 + ("pool",) * 2 + ("chain", "stem", "train", "infer", "dense", "dense", "stacks", "stacks"))
    dtype = rng.choice(("f32", "f32", "f32", "f64"))
    spread = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    while True:
        if kind == "conv":
            nd = rng.choice((1, 2, 2, 2, 3))
            w = tuple(rng.choice(((3, 5, 8, 9, 15), (1, 3, 3, 3, 5), (2, 3, 3))[nd - 1]) for _ in range(nd))
            s = tuple(rng.choice((1, 1, 1, 2)) for _ in range(nd))
            d = tuple(rng.choice((1, 1, 1, 2)) for _ in range(nd))
            p = tuple(rng.choice((0, 1)) * ((t - 1) * e // 2) for t, e in zip(w, d))
            grid = tuple(spread(*((64, 20000), (7, 128), (4, 48))[nd - 1]) for _ in range(nd))
            x = tuple((g - 1) * a + (t - 1) * e + 1 - 2 * q for g, a, t, e, q in zip(grid, s, w, d, p))
            case = _conv(None, dtype, spread(1, 128), spread(3, 320), spread(8, 512), x, w, s, p, d)
            del case["name"]
            if min(x) < 1:
                continue
        elif kind == "pool":
            nd = rng.choice((2, 2, 3))
            window, stride = rng.choice(((2, 2), (3, 2), (3, 3), (5, 1)))
            case = {"kind": kind, "dtype": dtype, "n": spread(1, 128), "c": spread(3, 256), "nd": nd, "g": spread(4, (112, 32)[nd - 2]),
                    "window": window, "stride": stride}
        elif kind == "chain":
            nd = rng.choice((2, 3))
            case = {"kind": kind, "dtype": dtype, "n": spread(1, 64), "c": spread(3, 96), "f": spread(8, 128), "nd": nd}
            case.update({"x" + a: 2 * spread(*((8, 64), (3, 32))[nd - 2]) for a in _AXES[:nd]})
        elif kind == "stem":
            case = {"kind": kind, "dtype": dtype, "n": spread(2, 64), "f": spread(16, 96), "p": spread(16, 64)}
        elif kind in ("train", "infer"):
            case = {"kind": kind, "dtype": dtype, "n": spread(*((16, 512) if kind == "train" else (1, 64))), "side": 4 * rng.randint(6, 16),
                    "c": rng.choice((1, 3)), "f1": spread(8, 48), "f2": spread(16, 96), "window": rng.choice((3, 5)), "classes": spread(10, 100)}
        elif kind == "dense":
            case = {"kind": kind, "dtype": dtype, "m": spread(32, 4096), "k": spread(64, 4096), "n": spread(32, 4096)}
        else:
            case = {"kind": kind, "dtype": dtype, "b": spread(2, 1024), "m": spread(16, 512), "k": spread(16, 512), "n": spread(16, 512)}
        cost = work(case)
        if cost["bytes"] < 6e8 and 1e4 < cost["flops"] + cost["bytes"] < (9e10 if dtype == "f32" else 3e10):
            return case


def _conv(name, dtype, n, c, f, x, w, stride, pad, dil):
    case = {"name": name, "kind": "conv", "dtype": dtype, "n": n, "c": c, "f": f, "nd": len(x)}
    for key, values in (("x", x), ("w", w), ("s", stride), ("p", pad), ("d", dil)):
        case.update({key + a: v for a, v in zip(_AXES, values)})
    return case


def _axes(case, key):
    return tuple(case[key + a] for a in _AXES[:case["nd"]])


def _conv_grid(case):
    return tuple((x + 2 * p - (w - 1) * d - 1) // s + 1 for x, w, s, p, d in zip(*(_axes(case, key) for key in "xwspd")))


def _pool_shapes(case):
    lead, nd = (case["n"], case["c"]), case["nd"]
    return (*lead, *((case["g"] - 1) * case["stride"] + case["window"],) * nd), (*lead, *(case["g"],) * nd)


def _net_filters(case):
    k, quarter = case["window"], case["side"] // 4
    return (case["f1"], case["c"], k, k), (case["f2"], case["f1"], k, k), (case["classes"], case["f2"], quarter, quarter)


# ------------------------------------------------------------------------------- what a program has in hand
class _Values:
    """Seeded values, made on the GPU: normal activations and gradients, filters scaled to keep the variance."""

    def __init__(self, case, seed):
        self._rng = torch.Generator(device="cuda").manual_seed(seed)
        self._dtype = case["dtype"]

    def host(self, shape, scale=1.0):
        values = torch.randn(shape, generator=self._rng, device="cuda", dtype=_TORCH[self._dtype])
        return values.mul_(scale).cpu().numpy()

    def filters(self, shape):
        return self.host(shape, (2.0 / np.prod(shape[1:])) ** 0.5)

    def device(self, shape, scale=1.0, constant=None):
        return mg.device_tensor(self.host(shape, scale), constant=constant)


def prepare(case, seed):
    values, kind = _Values(case, seed), case["kind"]
    state = {"case": case}
    if kind in ("conv", "chain"):
        nd, x = case["nd"], _axes(case, "x")
        filters = (case["f"], case["c"], *(_axes(case, "w") if kind == "conv" else (3,) * nd))
        grid = _conv_grid(case) if kind == "conv" else tuple(v // 2 for v in x)
        state["x"] = values.device((case["n"], case["c"], *x))
        state["w"] = mg.device_tensor(values.filters(filters))
        state["g"] = values.device((case["n"], case["f"], *grid), constant=True)
    elif kind == "pool":
        x, grid = _pool_shapes(case)
        state["x"], state["g"] = values.device(x), values.device(grid, constant=True)
    elif kind == "stem":
        n, f, p = case["n"], case["f"], case["p"]
        state["x"] = values.device((n, 3, 4 * p + 1, 4 * p + 1), constant=True)
        state["w"] = mg.device_tensor(values.filters((f, 3, 7, 7)))
        state["gamma"] = mg.device_tensor((1.0 + values.host((f,), 0.1)).astype(_NUMPY[case["dtype"]]))
        state["beta"] = values.device((f,), 0.1)
        state["g"] = values.device((n, f, p, p), constant=True)
    elif kind in ("train", "infer"):
        first, second, head = _net_filters(case)
        state["x"] = values.host((case["n"], case["c"], case["side"], case["side"]))
        state["params"] = [mg.tensor(values.filters(shape)) for shape in (first, second, head)]
        if kind == "train":
            state["params"] += [mg.tensor((1.0 + values.host((case["f1"],), 0.1)).astype(_NUMPY[case["dtype"]])), mg.tensor(values.host((case["f1"],), 0.1))]
            state["g"] = values.host((case["n"], case["classes"]), 1.0 / case["n"])
        else:
            state["params"] = [mg.device_tensor(p) for p in state["params"]]  # weights that stay as they are
    elif kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        state["a"], state["b"] = values.device((m, k)), values.device((k, n), k ** -0.5)
        state["g"] = values.device((m, n), constant=True)
    else:
        b, m, k, n = case["b"], case["m"], case["k"], case["n"]
        state["a"], state["b"] = values.device((b, m, k)), values.device((b, k, n), k ** -0.5)
        state["g"] = values.device((b, m, n), constant=True)
    return state


# ---------------------------------------------------------------------------------------------- one pass
class _OnDevice:
    """A result's device memory, described to torch; keeps the memory alive."""

    def __init__(self, array):
        self._array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str, "data": (array.buf.ptr, False), "version": 2}


def _whole(value):
    return value if isinstance(value, np.ndarray) else torch.as_tensor(_OnDevice(value), device="cuda")


def _results(outputs, leaves):
    """Values of `outputs` and gradients of `leaves`, where they are."""
    return [_whole(t._value) for t in outputs] + [_whole(t._grad) for t in leaves]


def _net(x, filters, window, scale=None):
    h = conv_nd(x, filters[0], stride=1, padding=window // 2)
    if scale is not None:
        h = batchnorm(h, gamma=scale[0], beta=scale[1], eps=1e-5)
    h = max_pool(relu(h), (2, 2), 2)
    h = max_pool(relu(conv_nd(h, filters[1], stride=1, padding=window // 2)), (2, 2), 2)
    return mg.einsum("nchw,kchw->nk", h, filters[2])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "conv":
        x, w = state["x"], state["w"]
        out = conv_nd(x, w, stride=_axes(case, "s"), padding=_axes(case, "p"), dilation=_axes(case, "d"))
        out.backward(state["g"])
        return _results((out,), (x, w))
    if kind == "chain":
        x, w, nd = state["x"], state["w"], case["nd"]
        pooled = max_pool(conv_nd(x, w, stride=1, padding=1), (2,) * nd, 2)
        loss = mg.sum(pooled * state["g"])
        loss.backward()
        return _results((pooled, loss), (x, w))
    if kind == "pool":
        x = state["x"]
        out = max_pool(x, (case["window"],) * case["nd"], case["stride"])
        out.backward(state["g"])
        return _results((out,), (x,))
    if kind == "stem":
        w, gamma, beta = state["w"], state["gamma"], state["beta"]
        out = max_pool(relu(batchnorm(conv_nd(state["x"], w, stride=2, padding=3), gamma=gamma, beta=beta, eps=1e-5)), (3, 3), 2)
        out.backward(state["g"])
        return _results((out,), (w, gamma, beta))
    if kind == "train":
        params = state["params"]
        logits = _net(mg.tensor(state["x"], constant=True), params[:3], case["window"], params[3:])
        loss = mg.sum(logits * state["g"])
        loss.backward()
        return [loss.data, logits.data] + [p.grad for p in params]
    if kind == "infer":
        with mg.no_autodiff:
            return _net(mg.tensor(state["x"]), state["params"], case["window"]).data
    a, b = state["a"], state["b"]
    out = a @ b
    out.backward(state["g"])
    return _results((out,), (a, b))


# -------------------------------------------------------------------------------- the same in 64 bits, by torch
def _conv64(x, w, stride, padding, dilation):
    """Correlation as one matrix product per tap of the window."""
    nd = x.ndim - 2
    x = torch.nn.functional.pad(x, [p for q in reversed(padding) for p in (q, q)])
    grid = [(a - (t - 1) * d - 1) // s + 1 for a, t, s, d in zip(x.shape[2:], w.shape[2:], stride, dilation)]
    out = 0.0
    for tap in np.ndindex(*w.shape[2:]):
        part = x[(slice(None), slice(None), *(slice(t * d, t * d + (g - 1) * s + 1, s) for t, d, g, s in zip(tap, dilation, grid, stride)))]
        out = out + w[(slice(None), slice(None), *tap)] @ part.transpose(0, 1).reshape(x.shape[1], -1)
    return out.reshape(w.shape[0], x.shape[0], *grid).transpose(0, 1)


def _pool64(x, window, stride):
    pool = {2: torch.nn.functional.max_pool2d, 3: torch.nn.functional.max_pool3d}[x.ndim - 2]
    return pool(x, window, stride)


def _batchnorm64(x, gamma, beta):
    axes = tuple(a for a in range(x.ndim) if a != 1)
    channel = lambda v: v.reshape(-1, *(1,) * (x.ndim - 2))
    mean = x.mean(axes, keepdim=True)
    var = ((x - mean) ** 2).mean(axes, keepdim=True)
    return channel(gamma) * (x - mean) / torch.sqrt(var + 1e-5) + channel(beta)


def _net64(x, filters, window, scale=None):
    same = ((1, 1), (window // 2,) * 2, (1, 1))
    h = _conv64(x, filters[0], *same)
    if scale is not None:
        h = _batchnorm64(h, *scale)
    h = _pool64(torch.relu(h), 2, 2)
    h = _pool64(torch.relu(_conv64(h, filters[1], *same)), 2, 2)
    return h.flatten(1) @ filters[2].flatten(1).T


def exact(case, seed):
    """What ``run`` returns, in 64 bits.  In float32 a gradient behind a maximum or a relu has no value in 64 bits to be
    held against: one window in some 100000 is decided the other way.  Nor has a loss that adds terms of either sign to
    nearly nothing; the values it is summed from are compared."""
    state, kind, decided = prepare(case, seed), case["kind"], case["dtype"] == "f64"

    def leaf(value, grad=True):
        value = value._value if isinstance(value, mg.Tensor) else value
        return torch.as_tensor(_whole(value), device="cuda").double().requires_grad_(grad)

    if kind in ("train", "infer"):
        x, params = leaf(state["x"], False), [leaf(p) for p in state["params"]]
        if kind == "infer":
            return _net64(x, params, case["window"]).detach()
        logits = _net64(x, params[:3], case["window"], params[3:])
        loss = (logits * leaf(state["g"], False)).sum()
        if decided:
            loss.backward()
        return [loss.detach() if decided else None, logits.detach()] + [p.grad for p in params]
    g = leaf(state["g"], False)
    if kind in ("conv", "chain"):
        leaves = x, w = leaf(state["x"]), leaf(state["w"])
        ones = (1,) * case["nd"]
        if kind == "conv":
            outputs = [_conv64(x, w, _axes(case, "s"), _axes(case, "p"), _axes(case, "d"))]
        else:
            outputs = [_pool64(_conv64(x, w, ones, ones, ones), 2, 2)]
            outputs.append((outputs[0] * g).sum())
    elif kind == "pool":
        leaves = (leaf(state["x"]),)
        outputs, decided = [_pool64(leaves[0], case["window"], case["stride"])], True
    elif kind == "stem":
        leaves = w, gamma, beta = leaf(state["w"]), leaf(state["gamma"]), leaf(state["beta"])
        outputs = [_pool64(torch.relu(_batchnorm64(_conv64(leaf(state["x"], False), w, (2, 2), (3, 3), (1, 1)), gamma, beta)), 3, 2)]
    else:
        leaves = leaf(state["a"]), leaf(state["b"])
        outputs = [leaves[0] @ leaves[1]]
    if decided or kind not in ("chain", "stem"):
        outputs[0].backward(g)
        grads = [t.grad for t in leaves]
    else:
        grads = [None] * len(leaves)
    if kind == "chain" and not decided:
        outputs[1] = None
    return [t if t is None else t.detach() for t in outputs] + grads


# ------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Operands read once and results written once; the arithmetic of the contractions."""
    kind, size = case["kind"], math.prod
    if kind in ("conv", "chain"):
        nd, x = case["nd"], _axes(case, "x")
        grid, taps = (_conv_grid(case), size(_axes(case, "w"))) if kind == "conv" else (x, 3 ** nd)
        xs, ws = case["n"] * case["c"] * size(x), case["f"] * case["c"] * taps
        outs = case["n"] * case["f"] * size(grid)
        flops = 6.0 * outs * case["c"] * taps
        count = 2 * (xs + ws) + 2 * (outs if kind == "conv" else outs // 2 ** nd)
    elif kind == "pool":
        x, grid = _pool_shapes(case)
        count, flops = 2 * (size(x) + size(grid)), 0.0
    elif kind == "stem":
        n, f, p = case["n"], case["f"], case["p"]
        flops = 4.0 * n * f * (2 * p + 1) ** 2 * 147
        count = n * 3 * (4 * p + 1) ** 2 + 2 * f * (147 + 2) + 2 * n * f * p * p
    elif kind in ("train", "infer"):
        n, s = case["n"], case["side"]
        filters = [size(shape) for shape in _net_filters(case)]
        products = n * (filters[0] * s * s + filters[1] * s * s // 4 + filters[2])
        flops = 2.0 * products if kind == "infer" else 6.0 * products - 2.0 * n * filters[0] * s * s
        count = n * case["c"] * s * s + (1 if kind == "infer" else 2) * sum(filters) + n * case["classes"]
    elif kind == "dense":
        m, k, n = case["m"], case["k"], case["n"]
        flops, count = 6.0 * m * k * n, 2 * (m * k + k * n + m * n)
    else:
        b, m, k, n = case["b"], case["m"], case["k"], case["n"]
        flops, count = 6.0 * b * m * k * n, 2 * b * (m * k + k * n + m * n)
    return {"bytes": float(count * _BYTES[case["dtype"]]), "flops": flops}


def tolerance(case):
    """Four times what the path was seen to differ by from ``exact`` (float64: filter gradients, sums over all positions,
    by 1.2e-14).  Pooling alone picks values and adds gradients in a fixed order.  In float32, the cases with a relu or a
    maximum behind a convolution may decide one element of millions the other way, which moves single gradients; nothing
    was seen to be decided otherwise in float64."""
    if case["kind"] == "pool":
        return "exact"
    if case["dtype"] == "f64":
        return {"rel": 5e-14, "max": 3e-13}
    return {"rel": 5e-3, "max": 0.1} if case["kind"] in ("chain", "stem", "train") else {"rel": 6e-6, "max": 3e-5}
