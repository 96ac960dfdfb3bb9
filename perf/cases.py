"""Performance cases: what a verification program does with this framework, from host bounds to host results.

A program holds a network (``NN``, weights resident after the first use) and the bounds of the inputs it wants
checked.  One pass builds the input set(s) from those bounds, runs ``NN.reach`` with a relax-star method at
relaxFactor = 1 and reads what it decides with: the output bounds, the verdict of a specification check, or the
bounds of every layer.  All of it is fp64, the only type the sets have.

The networks are random ones (Kaiming-normal weights, bias sigma 0.1) in the shapes of ``nnv_amd.configs`` and
their neighbours; a network depends on its sizes only, the inputs on the seed.

A case is a dict of

    net      layers, separated by blanks: fcN, convKxKxC[sS][pP], relu, bn, poolKxK[sS][pP], flatten, norm
    input    "784" (a vector) or "28x28x1" (an image, H x W x C)
    inputs   "boxes": every set is a box of half-width eps around a point of its own,
             "split": one such box bisected log2(sets) times, along its dimensions in turn,
             "general": one Star(V, C, d, lb, ub) with ``gens`` dense generators and ``cons`` constraint rows
    sets     how many sets are reached in one call (1: a single Star / ImageStar, not an array)
    eps      half-width of the box ("general": the size of what its generators add up to, per dimension)
    method   the relax-star variant
    want     "bounds", "robust" (NN.verify_robustness for the label the network gives the input) or
             "layers" (the bounds of every layer's output set)
"""
from __future__ import annotations

import functools
import math

import numpy as np

from nnv_amd import NN, ImageStar, Star
from nnv_amd.sets import Box

BIAS_SIGMA = 0.1


def _case(name, net, input, eps, sets=1, inputs="boxes", method="relax-star-area", want="bounds", gens=0, cons=0):
    c = {"net": net, "input": input, "inputs": inputs, "sets": sets, "eps": eps, "method": method, "want": want}
    if inputs == "general":
        c.update(gens=gens, cons=cons)
    return dict(c, name=name) if name else c


def _fc_net(widths):
    return " relu ".join("fc%d" % w for w in widths)


SMALL_NET = _fc_net([50] * 6 + [5])
WIDE_NET = _fc_net([1024] * 3 + [10])
CNN_28 = "conv3x3x16p1 relu conv3x3x32s2p1 relu fc100 relu fc10"
CNN_32 = "conv3x3x32p1 relu conv3x3x32s2 relu conv3x3x64p1 relu conv3x3x64s2 relu fc512 relu fc10"
CNN_NORM_POOL = "norm conv3x3x8p1 bn relu pool2x2s2 conv3x3x16p1 relu pool3x3s2p1 flatten fc32 relu fc10"


def listed():
    return [
        # a controller-sized network (5 inputs, 5 outputs), one query: latency
        _case("controller_one_box", SMALL_NET, "5", 0.02),
        # the same network under input splitting: one level of a branch-and-bound tree
        _case("controller_split_128", SMALL_NET, "5", 0.2, sets=128, inputs="split"),
        # an image classifier without convolutions, wide box: nearly every hidden neuron may change sign
        _case("fc_wide_box", WIDE_NET, "784", 0.02),
        # local robustness of the same classifier: a small box, few neurons change sign, half of them pass through
        _case("fc_robustness", WIDE_NET, "784", 0.0005, want="robust"),
        # a batch of test images, each with its own box
        _case("fc_100_images", WIDE_NET, "784", 1.0 / 255.0, sets=100),
        # branch and bound on the wide box: 1024 sub-boxes in one call
        _case("fc_split_1024", WIDE_NET, "784", 0.02, sets=1024, inputs="split"),
        # a small CNN, one image
        _case("cnn28_one_image", CNN_28, "28x28x1", 1.0 / 255.0),
        # the same with the bounds of every layer: which neurons are stable, where to split
        _case("cnn28_all_bounds", CNN_28, "28x28x1", 1.0 / 255.0, want="layers"),
        # the same, a batch of test images (an odd number)
        _case("cnn28_25_images", CNN_28, "28x28x1", 1.0 / 255.0, sets=25),
        # a deeper CNN on a colour image: the largest single set
        _case("cnn32_one_image", CNN_32, "32x32x3", 2.0 / 255.0),
        # input normalisation, batch normalisation, average pooling and a C-style flatten around the ReLU steps
        _case("cnn32_norm_pool", CNN_NORM_POOL, "32x32x3", 1.0 / 255.0),
        # a set that comes from elsewhere: dense generators, constraint rows, odd sizes
        _case("general_star", "fc700 relu fc700 relu fc20", "1000", 0.1, inputs="general", gens=1501, cons=50, want="layers"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(_log(rng, lo, hi)))))


def draw(rng):
    """One more case: a kind of work from the list above, its sizes spread over their range."""
    kind = rng.choice(["controller", "fc_one", "fc_robust", "fc_images", "fc_split", "cnn_one", "cnn_layers", "cnn_images",
                       "cnn_norm", "general"])
    method = rng.choice(["relax-star-area", "relax-star-area", "relax-star-bound", "relax-star-ub"])
    if kind == "controller":
        net = _fc_net([_logint(rng, 16, 200)] * rng.randint(2, 7) + [rng.randint(2, 9)])
        if rng.random() < 0.5:
            return _case("", net, str(rng.randint(3, 12)), round(_log(rng, 0.005, 0.1), 5), method=method)
        if rng.random() < 0.5:
            return _case("", net, str(rng.randint(8, 12)), round(_log(rng, 0.05, 0.3), 5), sets=2 ** rng.randint(1, 8),
                         inputs="split", method=method)
        return _case("", net, str(rng.randint(3, 12)), round(_log(rng, 0.005, 0.1), 5), sets=_logint(rng, 2, 200), method=method)
    if kind.startswith("fc_"):
        inp = str(_logint(rng, 100, 1000))
        net = _fc_net([_logint(rng, 200, 1100) for _ in range(rng.randint(2, 3))] + [rng.randint(2, 40)])
        if kind == "fc_one":
            return _case("", net, inp, round(_log(rng, 0.0005, 0.03), 6), method=method, want=rng.choice(["bounds", "bounds", "layers"]))
        if kind == "fc_robust":
            return _case("", net, inp, round(_log(rng, 0.0001, 0.0005), 6), method=method, want="robust")
        if kind == "fc_images":
            return _case("", net, inp, round(_log(rng, 0.0005, 0.01), 6), sets=_logint(rng, 2, 90), method=method)
        return _case("", net, inp, round(_log(rng, 0.005, 0.03), 6), sets=2 ** rng.randint(1, 9), inputs="split", method=method)
    if kind == "cnn_norm":
        hw = rng.randint(12, 32)
        net = "norm conv3x3x%dp1 bn relu pool2x2s2 conv3x3x%dp1 relu pool3x3s2p1 flatten fc%d relu fc%d" % (
            rng.randint(4, 8), rng.randint(6, 16), rng.randint(20, 64), rng.randint(2, 20))
        return _case("", net, "%dx%dx%d" % (hw, hw, rng.choice([1, 3])), round(_log(rng, 0.001, 0.008), 6), method=method)
    if kind == "general":
        net = "fc%d relu fc%d relu fc%d" % (_logint(rng, 100, 800), _logint(rng, 100, 800), rng.randint(2, 30))
        return _case("", net, str(_logint(rng, 100, 1000)), round(_log(rng, 0.01, 0.3), 5), inputs="general",
                     gens=_logint(rng, 50, 1500), cons=rng.randint(0, 60), method=method, want=rng.choice(["bounds", "layers"]))
    # the other CNNs
    sets = _logint(rng, 2, 24) if kind == "cnn_images" else 1
    deep = kind == "cnn_one" and rng.random() < 0.5
    h, w = (rng.randint(16, 32), rng.randint(16, 32)) if not deep else (rng.randint(20, 32),) * 2
    k = rng.choice([3, 3, 5])
    if deep:
        c1, c2 = rng.randint(8, 32), rng.randint(16, 64)
        net = "conv%dx%dx%dp1 relu conv3x3x%ds2 relu conv3x3x%dp1 relu conv3x3x%ds2 relu fc%d relu fc%d" % (
            k, k, c1, c1, c2, c2, _logint(rng, 50, 512), rng.randint(2, 20))
    else:
        net = "conv%dx%dx%dp%d relu conv3x3x%ds2p1 relu fc%d relu fc%d" % (
            k, k, rng.randint(4, 16), k // 2, rng.randint(8, 32), _logint(rng, 30, 200), rng.randint(2, 20))
    channels = rng.choice([1, 3]) if not sets > 8 else 1
    return _case("", net, "%dx%dx%d" % (h, w, channels), round(_log(rng, 0.001, 0.008), 6), sets=sets, method=method,
                 want="layers" if kind == "cnn_layers" else "bounds")


# ---- networks ---------------------------------------------------------------------------------------------------
def _shape(text):
    return tuple(int(x) for x in text.split("x"))


def _layer(word):
    """(kind, numbers) of one word of ``net``."""
    for kind in ("fc", "conv", "pool"):
        if word.startswith(kind):
            body, opts = word[len(kind):], {"s": 1, "p": 0}
            for key in ("p", "s"):
                if key in body:
                    body, value = body.rsplit(key, 1)
                    opts[key] = int(value)
            return kind, _shape(body), opts["s"], opts["p"]
    return word, (), 1, 0


@functools.lru_cache(maxsize=8)
def _network(net, input):
    """The program's network: built once, used for every input."""
    rs = np.random.RandomState(sum(ord(ch) * (i + 1) for i, ch in enumerate(net + input)))
    shape = _shape(input)
    dim = int(np.prod(shape))
    layers = []
    for word in net.split():
        kind, size, stride, pad = _layer(word)
        if kind == "fc":
            layers.append({"type": "fc", "W": rs.randn(size[0], dim) * math.sqrt(2.0 / dim), "b": rs.randn(size[0]) * BIAS_SIGMA})
            dim = size[0]
        elif kind == "conv":
            fan_in = size[0] * size[1] * shape[2]
            layers.append({"type": "conv", "W": rs.randn(size[0], size[1], shape[2], size[2]) * math.sqrt(2.0 / fan_in),
                           "b": rs.randn(size[2]) * BIAS_SIGMA, "padding": [pad] * 4, "stride": [stride] * 2, "dilation": [1, 1]})
        elif kind == "pool":
            layers.append({"type": "avgpool", "pool": list(size), "stride": [stride] * 2, "padding": [pad] * 4})
        elif kind == "relu":
            layers.append({"type": "relu"})
        elif kind == "bn":
            c = shape[2]
            layers.append({"type": "batchnorm", "mean": 0.1 * rs.randn(c), "var": rs.rand(c) + 0.5, "eps": 1e-5,
                           "scale": 1.0 + 0.1 * rs.randn(c), "offset": 0.1 * rs.randn(c)})
        elif kind == "norm":
            c = shape[2]
            layers.append({"type": "imageinput", "normalization": "zscore", "input_size": list(shape),
                           "mean": rs.rand(1, 1, c), "std": 0.5 + rs.rand(c)})
        elif kind == "flatten":
            layers.append({"type": "flatten", "flatten_type": "nnet.keras.layer.FlattenCStyleLayer"})
        else:
            raise ValueError("unknown layer %r" % word)
        shape, dim = _after(kind, size, stride, pad, shape, dim)
    return NN.from_config(layers)


def _after(kind, size, stride, pad, shape, dim):
    """Image shape and dimension behind a layer."""
    if kind in ("conv", "pool"):
        h, w = ((x + 2 * pad - k) // stride + 1 for x, k in zip(shape[:2], size[:2]))
        shape = (h, w, size[2] if kind == "conv" else shape[2])
        return shape, h * w * shape[2]
    if kind == "fc":
        return shape, size[0]
    return shape, dim


def _confident_point(net, rs, dim):
    """Of a few points the one whose label the network is surest of: what a robustness check starts from."""
    best = None
    for _ in range(16):
        x = rs.rand(dim)
        y = x
        for layer in net.Layers:
            y = layer.evaluate(y)
        top = np.sort(y)
        if best is None or top[-1] - top[-2] > best[0]:
            best = (top[-1] - top[-2], x, int(np.argmax(y)))
    return best[1], best[2]


# ---- a pass -----------------------------------------------------------------------------------------------------
def prepare(case, seed):
    net = _network(case["net"], case["input"])
    shape = _shape(case["input"])
    dim = int(np.prod(shape))
    rs = np.random.RandomState(seed % (1 << 32))
    state = {"net": net, "shape": shape, "want": case["want"], "sets": case["sets"],
             "options": {"reachMethod": case["method"], "relaxFactor": 1}}
    eps = case["eps"]
    if case["inputs"] == "general":
        gens, cons = case["gens"], case["cons"]
        V = np.concatenate([rs.rand(dim, 1), rs.randn(dim, gens) * (eps / gens)], axis=1)
        # constraint rows that cut corners off the predicate box (a = 0 stays feasible)
        C, d = rs.randn(cons, gens), (0.5 + rs.rand(cons)) * math.sqrt(gens)
        if not cons:
            C, d = np.zeros((1, gens)), np.zeros(1)
        state["star"] = Star(V, C, d, -np.ones(gens), np.ones(gens))
        return state
    if case["want"] == "robust":
        x, state["label"] = _confident_point(net, rs, dim)
        state["lb"], state["ub"] = x - eps, x + eps
    elif case["inputs"] == "split":
        x = rs.rand(dim)
        cuts = case["sets"].bit_length() - 1
        state["lb"], state["ub"] = Box(x - eps, x + eps).partition_bounds([i % dim for i in range(cuts)], [2] * cuts)
    else:
        x = rs.rand(dim, case["sets"]) if case["sets"] > 1 else rs.rand(dim)
        state["lb"], state["ub"] = np.asfortranarray(x - eps), np.asfortranarray(x + eps)
    return state


def _input_set(state):
    if "star" in state:
        return state["star"]
    lb, ub, shape = state["lb"], state["ub"], state["shape"]
    if state["sets"] > 1:
        if len(shape) == 1:
            return Star.from_boxes(lb, ub)
        return [ImageStar(lb[:, i].reshape(shape, order="F"), ub[:, i].reshape(shape, order="F")) for i in range(state["sets"])]
    if len(shape) == 1:
        return Star(lb, ub)
    return ImageStar(lb.reshape(shape, order="F"), ub.reshape(shape, order="F"))


def run(state):
    net = state["net"]
    if state["want"] == "robust":
        verdict = net.verify_robustness(_input_set(state), state["options"], state["label"])
        return (verdict,) + net.reachSet[-1].estimateRanges()
    out = net.reach(_input_set(state), state["options"])
    if state["want"] == "layers":
        return [s.estimateRanges() for s in net.reachSet]
    return out.estimateRanges() if state["sets"] == 1 else Star.estimateRanges_array(out)


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def work(case):
    """Weights and input bounds read once, the output set written once; the products of the weights with the centres,
    with the vectors the range estimates need, and with the generator columns that are not images of a single input
    entry, over the rows a ReLU passes through and (in the convolutional part) inside the columns' windows.

    How many neurons change sign is estimated from the box: a first-layer pre-activation has standard deviation 0.8
    and a half-width of 1.13 eps sqrt(fan-in); every neuron that changes sign widens the layers behind it."""
    shape, sets = _shape(case["input"]), case["sets"]
    dim = int(np.prod(shape))
    image = len(shape) == 3
    general = case["inputs"] == "general"
    width, crossing, passed = case["eps"], 1.0, 1.0       # half-width of the layer's input, shares of its rows
    dense = float(case["gens"]) if general else 0.0        # generator columns that are not unit vectors
    units = 0.0 if general else float(dim)                 # ... and that are
    window = math.inf if general else 1.0                  # positions a dense column reaches
    live = 1.0
    flops = bytes_ = 0.0
    first = True
    for word in case["net"].split():
        kind, size, stride, pad = _layer(word)
        if kind in ("fc", "conv"):
            if kind == "fc":
                out, taps, positions, weights = size[0], dim, 1.0, size[0] * dim
                reach = 1.0
            else:
                h, w = ((x + 2 * pad - k) // stride + 1 for x, k in zip(shape[:2], size[:2]))
                taps, weights, positions = size[0] * size[1] * shape[2], size[0] * size[1] * shape[2] * size[2], h * w
                out = h * w * size[2]
                window = min(float(positions), (math.sqrt(window) + size[0] - 1) ** 2 / stride ** 2)
                reach = window
            channels = out / positions
            flops += sets * 2.0 * channels * taps * live * (positions + dense * reach)       # centre and dense columns
            flops += sets * 2.0 * 2.0 * channels * min(taps, units) * (positions if kind == "conv" else 1.0)  # ranges of the unit columns
            flops += sets * 4.0 * dense * reach * channels                                   # ranges of the dense columns
            bytes_ += 8.0 * (weights + channels)
            dense, units = dense + units, 0.0
            grow = 1.13 * math.sqrt(taps)
            width = width * grow if first and not general else width * (1.0 + 0.5 * crossing * grow) if not first else 1.13 * width
            first = False
        elif kind == "relu":
            crossing = math.erf(min(width / (0.8 * math.sqrt(2.0)), 6.0))
            passed = 0.5 * (1.0 - crossing)
            live, units = passed, crossing * dim
        elif kind in ("bn", "norm", "pool", "flatten"):
            columns = dense if kind != "norm" else units
            flops += sets * 2.0 * dim * (columns if math.isinf(window) else columns * min(1.0, window / max(1, shape[0] * shape[1])))
            if kind == "pool":
                window = max(1.0, window / stride ** 2)
                live, crossing = 1.0, crossing * 0.5
                dense, units = dense + units, 0.0
        shape, dim = _after(kind, size, stride, pad, shape, dim)
        bytes_ += 2 * 8.0 * dim if case["want"] == "layers" else 0.0
    n = dense + units
    bytes_ += sets * 8.0 * dim * (n + 1.0) + sets * 2 * 8.0 * dim
    bytes_ += 8.0 * int(np.prod(_shape(case["input"]))) * ((case["gens"] + 1) if general else 2 * sets)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """fp64 throughout: the same reach with its products formed densely, or with its sums in another order, differs
    from the default by up to 2.4e-15 of the results' norm (measured over these cases and 26 drawn ones)."""
    return {"rel": 1e-14, "max": 1e-13}
