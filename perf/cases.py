"""The work this framework is used for, as cases that can be timed and compared.

Every case goes through the Python front end (jittor_amd): operands that lie in device memory as Vars, a graph built by
the ordinary functions, `jt.grad` where the case trains, one `jt.sync` of what the program asks for.  The results are
handed out as torch tensors that look at the Vars' device buffers (no copy, no wait).

A case is a dict: "kind" names the family, the other entries are its sizes, its data type and its options.
"""
import math

import torch

import jittor_amd as jt

_TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16, "int32": torch.int32}
_TYPESTR = {"float32": "<f4", "float16": "<f2", "bfloat16": "<i2", "int32": "<i4"}
_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2, "int32": 4}


# ---- torch <-> Var ------------------------------------------------------------------------------------------------
def _var(t, dtype):
    """A Var with the values of a torch tensor (in storage format: bfloat16 travels as its bits)."""
    t = t.to(_TORCH[dtype]).contiguous()
    if dtype == "bfloat16":
        return jt.from_storage(t.view(torch.int16).cpu().numpy().view("uint16"), dtype)
    return jt.from_storage(t.cpu().numpy(), dtype)


class _Device:
    """A computed Var's device buffer under the array interface that torch takes; keeps the Var alive."""

    def __init__(self, v):
        self.v = v
        self.__cuda_array_interface__ = {"shape": tuple(v.shape), "typestr": _TYPESTR[v.dtype], "data": (v.raw_ptr(), False),
                                         "strides": None, "version": 2}


def _out(v):
    t = torch.as_tensor(_Device(v), device="cuda")
    return t.view(torch.bfloat16) if v.dtype == "bfloat16" else t


def _finish(outs):
    """Computes the named results in one sync and hands them out."""
    jt.sync(list(outs.values()))
    return {k: _out(v) for k, v in outs.items()}


class _Maker:
    """Inputs from a seed alone, made on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))
        self.dtype = dtype
        self.made = {}

    def normal(self, name, shape, scale=1.0, shift=0.0, dtype=None):
        t = torch.randn(list(shape), generator=self.g, device="cuda") * scale + shift
        self.made[name] = _var(t, dtype or self.dtype)

    def uniform(self, name, shape, lo=0.0, hi=1.0):
        t = torch.rand(list(shape), generator=self.g, device="cuda") * (hi - lo) + lo
        self.made[name] = _var(t, self.dtype)

    def done(self):
        jt.sync(list(self.made.values()))                  # uploads them
        return self.made


def _conv_out(c):
    p = c["k"] // 2
    return (c["size"] + 2 * p - c["k"]) // c["stride"] + 1


def _conv_flops(n, cin, cout, o, k):
    return 2.0 * n * cout * o * o * cin * k * k


# ---- the listed cases ---------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest training step a user runs: a small float32 CNN with a linear head and cross entropy at batch 4; its
        # tensors are a few KB, so what it costs is graph, dispatch and launches
        {"name": "step_small_cnn", "kind": "small_cnn", "n": 4, "cin": 8, "size": 12, "width": 16, "classes": 5, "dtype": "float32"},
        # ResNet-50's stage-3 bottleneck block (the stage with most blocks) at batch 64 in bfloat16: 1x1, 3x3, 1x1 convolutions,
        # relu, shortcut, forward and every gradient
        {"name": "step_bottleneck", "kind": "bottleneck", "n": 64, "c": 1024, "mid": 256, "size": 14, "dtype": "bfloat16"},
        # a ResNet's stem in Jittor's default type: 7x7 convolution of stride 2 on images, relu, 3x3 max pooling of stride 2, forward
        # and the gradient of the weights (images have none)
        {"name": "step_stem_f32", "kind": "stem", "n": 32, "size": 224, "width": 64, "dtype": "float32"},
        # inference through a wide 3x3 layer: the meta-operator convolution at its largest
        {"name": "conv3x3_infer", "kind": "conv", "train": False, "n": 64, "cin": 256, "cout": 512, "size": 28, "k": 3, "stride": 1, "dtype": "bfloat16"},
        # the strided 3x3 layer between two stages, forward and both gradients
        {"name": "conv3x3_s2_train", "kind": "conv", "train": True, "n": 64, "cin": 256, "cout": 256, "size": 28, "k": 3, "stride": 2, "dtype": "bfloat16"},
        # a depthwise 3x3 layer (one channel per group), forward and both gradients, float32
        {"name": "depthwise_train", "kind": "depthwise", "n": 32, "c": 128, "size": 56, "k": 3, "stride": 1, "dtype": "float32"},
        # image to columns by reindex: 3x3 windows of stride 1 with padding 1
        {"name": "im2col", "kind": "im2col", "n": 32, "c": 64, "size": 56, "k": 3, "stride": 1, "dtype": "float32"},
        # scatter-add of values into bins by index (histograms, the gradient of an embedding or a gather); indices as they come in
        # earnest, a few bins taking most of them (bounded Zipf)
        {"name": "scatter_add", "kind": "scatter", "n": 1 << 24, "bins": 1 << 20, "op": "add", "zipf": True, "dtype": "float32"},
        # a chain of element-wise ops with broadcast scale and bias that the fuser makes one kernel of
        {"name": "fused_chain", "kind": "chain", "a": 64, "b": 512, "c": 1024, "dtype": "float32"},
        # a plain sum along the innermost axis
        {"name": "reduce_sum", "kind": "reduce", "a": 1, "b": 8192, "c": 4096, "axis": 2, "op": "add", "dtype": "float32"},
        # layer normalisation with scale and shift, forward and all gradients: reductions and element-wise passes over one tensor
        {"name": "layernorm_train", "kind": "layernorm", "rows": 16384, "cols": 1024, "dtype": "float32"},
        # a linear layer with bias, forward and all gradients, in Jittor's default type
        {"name": "linear_train", "kind": "linear", "m": 2048, "k": 1024, "n": 1024, "dtype": "float32"},
    ]


# ---- other cases of the same ranges -------------------------------------------------------------------------------
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case.  Sizes are spread over the logarithm of their ranges; half of the channel counts and extents are round
    numbers, as models have them, the others any number."""
    kind = rng.choice(["small_cnn", "bottleneck", "stem", "conv", "conv", "depthwise", "im2col", "scatter", "chain", "reduce",
                       "layernorm", "softmax", "linear"])

    def channels(lo, hi):
        c = _log(rng, lo, hi)
        return max(lo, c // 16 * 16) if rng.random() < 0.5 and c >= 16 else c

    if kind == "small_cnn":
        return {"kind": kind, "n": _log(rng, 1, 64), "cin": rng.randint(1, 16), "size": rng.randint(8, 40), "width": rng.randint(8, 48),
                "classes": rng.randint(2, 100), "dtype": "float32"}
    if kind == "bottleneck":
        c, mid, size = rng.choice([(1024, 256, 14), (1024, 256, 14), (2048, 512, 7)])
        return {"kind": kind, "n": _log(rng, 1, 64), "c": c, "mid": mid, "size": size, "dtype": rng.choice(["bfloat16", "bfloat16", "float32"])}
    if kind == "stem":
        return {"kind": kind, "n": _log(rng, 1, 32), "size": rng.choice([64, 96, 128, 160, 192, 224, rng.randint(48, 224)]),
                "width": channels(16, 64), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
    if kind == "conv":
        while True:
            # inference: maps of a CIFAR network or of a ResNet's stages behind the first; training: its late stages and the strided
            # layers in front of them
            c = {"kind": kind, "train": rng.random() < 0.6, "n": _log(rng, 1, 64), "cin": channels(16, 512), "cout": channels(16, 512),
                 "k": rng.choice([1, 3, 3, 3, 5]), "stride": rng.choice([1, 1, 2]), "dtype": rng.choice(["bfloat16", "bfloat16", "float16", "float32"])}
            c["size"] = rng.choice([7, 14, rng.randint(9, 15)] if c["train"] and c["stride"] == 1 else [7, 14, 28, 32, rng.randint(7, 32)])
            o = _conv_out(c)
            flops = _conv_flops(c["n"], c["cin"], c["cout"], o, c["k"]) * (3 if c["train"] else 1)
            elements = c["n"] * (c["cin"] * c["size"] ** 2 + c["cout"] * o * o)
            if flops <= (6e10 if c["dtype"] != "float32" else 3e9) and elements <= 5e7:
                return c
    if kind == "depthwise":
        while True:
            c = {"kind": kind, "n": _log(rng, 1, 64), "c": channels(16, 512), "size": rng.choice([7, 14, 28, 56, 112, rng.randint(7, 112)]),
                 "k": rng.choice([3, 3, 5]), "stride": rng.choice([1, 1, 2]), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
            if c["n"] * c["c"] * c["size"] ** 2 <= 12900000:
                return c
    if kind == "im2col":
        while True:
            c = {"kind": kind, "n": _log(rng, 1, 64), "c": channels(3, 256), "size": rng.randint(7, 112), "k": rng.choice([2, 3, 3, 5]),
                 "stride": rng.choice([1, 1, 2]), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
            if c["n"] * c["c"] * (_conv_out(c) * c["k"]) ** 2 <= 58000000:
                return c
    if kind == "scatter":
        return {"kind": kind, "n": _log(rng, 1 << 12, 1 << 24), "bins": _log(rng, 1 << 8, 1 << 20), "op": rng.choice(["add", "add", "maximum"]),
                "zipf": rng.random() < 0.6, "dtype": "float32"}
    if kind == "chain":
        while True:
            c = {"kind": kind, "a": _log(rng, 1, 256), "b": _log(rng, 1, 1024), "c": _log(rng, 8, 4096), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
            if 4096 <= c["a"] * c["b"] * c["c"] <= 33600000:
                return c
    if kind == "reduce":
        while True:
            c = {"kind": kind, "a": _log(rng, 1, 256), "b": _log(rng, 4, 65536), "c": _log(rng, 4, 8192), "axis": rng.choice([0, 1, 2, 2, 3]),
                 "op": rng.choice(["add", "add", "mean", "maximum"]), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
            if 16384 <= c["a"] * c["b"] * c["c"] <= 33600000:
                return c
    if kind in ("layernorm", "softmax"):
        while True:
            c = {"kind": kind, "rows": _log(rng, 16, 65536), "cols": _log(rng, 32, 16384), "dtype": rng.choice(["float32", "float32", "bfloat16"])}
            if 16384 <= c["rows"] * c["cols"] <= 8300000:
                return c
    while True:
        c = {"kind": "linear", "m": _log(rng, 1, 8192), "k": channels(16, 4096), "n": channels(16, 4096), "dtype": rng.choice(["float32", "float32", "bfloat16", "float16"])}
        if c["m"] * c["k"] * c["n"] <= (2.1e9 if c["dtype"] == "float32" else 2.5e8):
            return c


# ---- inputs -------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    c = dict(case)
    kind, m = c["kind"], _Maker(seed, c["dtype"])
    if kind == "small_cnn":
        w = c["width"]
        m.normal("x", [c["n"], c["cin"], c["size"], c["size"]])
        m.normal("w1", [w, c["cin"], 3, 3], math.sqrt(2.0 / (9 * c["cin"])))
        m.normal("w2", [w, w, 3, 3], math.sqrt(2.0 / (9 * w)))
        m.normal("wl", [c["classes"], w], math.sqrt(1.0 / w))
        m.normal("bl", [c["classes"]], 0.1)
        label = torch.randint(0, c["classes"], [c["n"]], generator=m.g, device="cuda")
        m.made["onehot"] = _var(torch.nn.functional.one_hot(label, c["classes"]), "float32")
    elif kind == "bottleneck":
        x = [c["n"], c["c"], c["size"], c["size"]]
        m.normal("x", x)
        m.normal("w1", [c["mid"], c["c"], 1, 1], math.sqrt(2.0 / c["c"]))
        m.normal("w2", [c["mid"], c["mid"], 3, 3], math.sqrt(2.0 / (9 * c["mid"])))
        m.normal("w3", [c["c"], c["mid"], 1, 1], math.sqrt(2.0 / c["mid"]))
        m.normal("g", x)                                   # what the layers behind the block send back
    elif kind == "stem":
        o = ((c["size"] - 1) // 2 + 1 + 2 - 3) // 2 + 1
        m.normal("x", [c["n"], 3, c["size"], c["size"]])
        m.normal("w", [c["width"], 3, 7, 7], math.sqrt(2.0 / 147))
        m.normal("g", [c["n"], c["width"], o, o])
    elif kind in ("conv", "depthwise"):
        cin, cout = (c["cin"], c["cout"]) if kind == "conv" else (c["c"], c["c"])
        per = cin if kind == "conv" else 1
        m.normal("x", [c["n"], cin, c["size"], c["size"]])
        m.normal("w", [cout, per, c["k"], c["k"]], math.sqrt(2.0 / (per * c["k"] ** 2)))
        if kind == "depthwise" or c["train"]:
            m.normal("g", [c["n"], cout, _conv_out(c), _conv_out(c)])
    elif kind == "im2col":
        m.normal("x", [c["n"], c["c"], c["size"], c["size"]])
    elif kind == "scatter":
        m.uniform("v", [c["n"]])
        if c["zipf"]:
            weight = torch.arange(1, c["bins"] + 1, dtype=torch.float64, device="cuda") ** -1.1
            cdf = torch.cumsum(weight, 0) / weight.sum()
            u = torch.rand([c["n"]], dtype=torch.float64, generator=m.g, device="cuda")
            index = torch.searchsorted(cdf, u).clamp_(max=c["bins"] - 1)
        else:
            index = torch.randint(0, c["bins"], [c["n"]], generator=m.g, device="cuda")
        m.made["index"] = _var(index, "int32")
    elif kind == "chain":
        m.normal("x", [c["a"], c["b"], c["c"]])
        m.normal("scale", [c["b"], 1])
        m.normal("bias", [1, c["c"]])
    elif kind == "reduce":
        m.uniform("x", [c["a"], c["b"], c["c"]], -1.0, 1.0)
    elif kind == "layernorm":
        m.normal("x", [c["rows"], c["cols"]], 1.5, 0.3)
        m.normal("gamma", [c["cols"]], 0.2, 1.0)
        m.normal("beta", [c["cols"]], 0.2)
        m.normal("g", [c["rows"], c["cols"]])
    elif kind == "softmax":
        m.normal("x", [c["rows"], c["cols"]], 2.0)
        m.normal("g", [c["rows"], c["cols"]])
    elif kind == "linear":
        m.normal("x", [c["m"], c["k"]])
        m.normal("w", [c["n"], c["k"]], math.sqrt(1.0 / c["k"]))
        m.normal("b", [c["n"]], 0.1)
        m.normal("g", [c["m"], c["n"]])
    else:
        raise ValueError("unknown kind %r" % kind)
    return {"case": c, "in": m.done()}


# ---- one pass -----------------------------------------------------------------------------------------------------
def _small_cnn(c, v):
    h = jt.nn.relu(jt.nn.conv2d(v["x"], v["w1"], padding=1))
    h = jt.nn.max_pool2d(h, 3, 2, 1)
    h = jt.nn.relu(jt.nn.conv2d(h, v["w2"], stride=2, padding=1))
    logits = jt.nn.linear(h.mean([2, 3]), v["wl"], v["bl"])
    shifted = logits - logits.max([1], keepdims=True)
    logp = shifted - shifted.exp().sum([1], keepdims=True).log()
    loss = (logp * v["onehot"]).sum() * (-1.0 / c["n"])
    names = ["w1", "w2", "wl", "bl"]
    grads = jt.grad(loss, [v[k] for k in names])
    return dict({"loss": loss, "logits": logits}, **{"d" + k: g for k, g in zip(names, grads)})


def _with_grads(y, v, names):
    """The result and the gradients of the named operands, `g` being what arrives at the result."""
    grads = jt.grad((y * v["g"]).sum(), [v[k] for k in names])
    return dict({"y": y}, **{"d" + k: g for k, g in zip(names, grads)})


def _bottleneck(c, v):
    h = jt.nn.relu(jt.nn.conv2d(v["x"], v["w1"]))
    h = jt.nn.relu(jt.nn.conv2d(h, v["w2"], padding=1))
    h = jt.nn.conv2d(h, v["w3"])
    return _with_grads(jt.nn.relu(h + v["x"]), v, ["x", "w1", "w2", "w3"])


def _stem(c, v):
    h = jt.nn.relu(jt.nn.conv2d(v["x"], v["w"], stride=2, padding=3))
    return _with_grads(jt.nn.max_pool2d(h, 3, 2, 1), v, ["w"])


def _conv(c, v):
    y = jt.nn.conv2d(v["x"], v["w"], stride=c["stride"], padding=c["k"] // 2)
    return _with_grads(y, v, ["x", "w"]) if c["train"] else {"y": y}


def _depthwise(c, v):
    y = jt.nn.conv2d(v["x"], v["w"], stride=c["stride"], padding=c["k"] // 2, groups=c["c"])
    return _with_grads(y, v, ["x", "w"])


def _im2col(c, v):
    p, s, o = c["k"] // 2, c["stride"], _conv_out(c)
    return {"y": v["x"].reindex([c["n"], c["c"], o, o, c["k"], c["k"]], ["i0", "i1", "i2*%d+i4-%d" % (s, p), "i3*%d+i5-%d" % (s, p)])}


def _scatter(c, v):
    return {"y": v["v"].reindex_reduce(c["op"], [c["bins"]], ["@e0(i0)"], extras=[v["index"]])}


def _chain(c, v):
    x = v["x"]
    return {"y": (-jt.nn.relu(x * v["scale"] + v["bias"])).exp() * x.sigmoid()}


def _reduce(c, v):
    return {"y": v["x"].reduce(c["op"], [] if c["axis"] == 3 else [c["axis"]])}          # axis 3: over everything


def _layernorm(c, v):
    d = v["x"] - v["x"].mean([1], keepdims=True)
    y = d / ((d * d).mean([1], keepdims=True) + 1e-5).sqrt() * v["gamma"] + v["beta"]
    return _with_grads(y, v, ["x", "gamma", "beta"])


def _softmax(c, v):
    e = (v["x"] - v["x"].max([1], keepdims=True)).exp()
    return _with_grads(e / e.sum([1], keepdims=True), v, ["x"])


def _linear(c, v):
    return _with_grads(jt.nn.linear(v["x"], v["w"], v["b"]), v, ["x", "w", "b"])


_RUN = {"small_cnn": _small_cnn, "bottleneck": _bottleneck, "stem": _stem, "conv": _conv, "depthwise": _depthwise, "im2col": _im2col,
        "scatter": _scatter, "chain": _chain, "reduce": _reduce, "layernorm": _layernorm, "softmax": _softmax, "linear": _linear}


def run(state):
    c = state["case"]
    return _finish(_RUN[c["kind"]](c, state["in"]))


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def work(case):
    """Bytes: every operand read once and every result written once.  Flops: multiply-adds of convolutions and products counted
    twice; a handful per element for the others."""
    c = dict(case)
    kind, e = c["kind"], _BYTES[c["dtype"]]
    if kind == "small_cnn":
        s, w = c["size"], c["width"]
        s2 = (s - 1) // 2 + 1
        s3 = (s2 - 1) // 2 + 1
        weights = w * c["cin"] * 9 + w * w * 9 + c["classes"] * (w + 1)
        flops = 2 * _conv_flops(c["n"], c["cin"], w, s, 3) + 3 * _conv_flops(c["n"], w, w, s3, 3) + 6.0 * c["n"] * w * c["classes"]
        return {"bytes": e * (c["n"] * c["cin"] * s * s + 2 * weights + 2 * c["n"] * c["classes"] + 1), "flops": flops}
    if kind == "bottleneck":
        big = c["n"] * c["c"] * c["size"] ** 2
        weights = 2 * c["c"] * c["mid"] + 9 * c["mid"] ** 2
        return {"bytes": e * (4.0 * big + 2 * weights), "flops": 6.0 * c["n"] * c["size"] ** 2 * weights}
    if kind == "stem":
        o = (c["size"] - 1) // 2 + 1
        p = (o - 1) // 2 + 1
        return {"bytes": e * (3.0 * c["n"] * c["size"] ** 2 + 2 * 147 * c["width"] + 2 * c["n"] * c["width"] * p * p),
                "flops": 2 * _conv_flops(c["n"], 3, c["width"], o, 7)}
    if kind in ("conv", "depthwise"):
        o = _conv_out(c)
        cin, cout, per = (c["cin"], c["cout"], c["cin"]) if kind == "conv" else (c["c"], c["c"], 1)
        x, y, w = c["n"] * cin * c["size"] ** 2, c["n"] * cout * o * o, cout * per * c["k"] ** 2
        both = 2 if kind == "depthwise" or c["train"] else 1
        return {"bytes": float(e * both * (x + y + w)), "flops": _conv_flops(c["n"], per, cout, o, c["k"]) * (3 if both == 2 else 1)}
    if kind == "im2col":
        x, y = c["n"] * c["c"] * c["size"] ** 2, c["n"] * c["c"] * (_conv_out(c) * c["k"]) ** 2
        return {"bytes": float(e * (x + y)), "flops": 0.0}
    if kind == "scatter":
        return {"bytes": 8.0 * c["n"] + 4.0 * c["bins"], "flops": float(c["n"])}
    if kind == "chain":
        n = c["a"] * c["b"] * c["c"]
        return {"bytes": float(e * (2 * n + c["b"] + c["c"])), "flops": 10.0 * n}
    if kind == "reduce":
        n = c["a"] * c["b"] * c["c"]
        kept = 1 if c["axis"] == 3 else n // (c["a"], c["b"], c["c"])[c["axis"]]
        return {"bytes": float(e * (n + kept)), "flops": float(n)}
    if kind == "layernorm":
        n = c["rows"] * c["cols"]
        return {"bytes": float(e * (4 * n + 4 * c["cols"])), "flops": 20.0 * n}
    if kind == "softmax":
        n = c["rows"] * c["cols"]
        return {"bytes": float(e * 4 * n), "flops": 12.0 * n}
    x, w, y = c["m"] * c["k"], c["n"] * c["k"], c["m"] * c["n"]
    return {"bytes": float(e * (2 * x + 2 * w + 2 * y + 2 * c["n"])), "flops": 6.0 * c["m"] * c["k"] * c["n"]}


def tolerance(case):
    """What another correct implementation of the same precision may be off by: about four times what these paths show against the same
    graph in 64 bits (single precision: up to 1.1e-6 for products and convolutions, 2e-7 elsewhere; half precision: 3e-3 for one rounding,
    9e-3 for a block's result).  A relu or a maximum that decides the other way where its operands agree to the last bit sends a whole
    gradient elsewhere, which shows in steps that have them: 1.1e-3 in the weights' gradient of the stem, more in half precision."""
    kind, half = case["kind"], case["dtype"] != "float32"
    if kind == "im2col" or kind in ("reduce", "scatter") and case["op"] == "maximum":
        return "exact"
    if half:
        return {"rel": 0.03, "max": 0.99}
    if kind in ("stem", "bottleneck", "small_cnn"):
        return {"rel": 5e-3, "max": 0.99}
    return {"rel": 5e-6, "max": 5e-4}
