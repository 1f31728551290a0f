"""What the speed of this framework is measured on: passes through its Python classes as a program that computes
with arrays calls them.

A case is a kind of work, an element type and a shape. The kinds are the chains that the benchmark and the tests
of this repository are made of (vector updates, broadcasting, axis reductions, strided views, softmax and layer
normalisation along rows) and what stands around them in a program that prepares data and looks at results
(standardised columns, masks and selections, running sums, functions, logic on bits). Arrays come from the
library's pool and are filled on the device; results come back as tensors that view the library's own memory, so
nothing is copied to look at them.

Bytes are counted call by call: each call of the chain reads its operands once and writes its result once, since
the caller may hold every one of those results.
"""
import math

import numpy as np
import torch

from cumo_amd import Bit, DFloat, Fused, Int32, NMath, SFloat

CLASS = {"SFloat": SFloat, "DFloat": DFloat, "Int32": Int32}
SIZE = {"SFloat": 4, "DFloat": 8, "Int32": 4}


def listed():
    return [
        # one step of an iterative method on a short vector (the reference's smallest benchmark size): launches
        {"name": "step 10000", "kind": "step", "type": "SFloat", "shape": "10000"},
        # the same step on the benchmark's first vector, 2^20 elements
        {"name": "step 2^20", "kind": "step", "type": "SFloat", "shape": "1048576"},
        # sums and extremes of a small matrix, whole and along either axis (the reference's reduction benchmark)
        {"name": "reduce 500x500", "kind": "reduce", "type": "SFloat", "shape": "500x500"},
        # the same of an activation-sized tensor, axes first, middle and last
        {"name": "reduce 64x512x1024", "kind": "reduce", "type": "SFloat", "shape": "64x512x1024"},
        # a bias row added to a matrix in double precision, row sums and row maxima of the result
        {"name": "bias 4096x4096", "kind": "bias", "type": "DFloat", "shape": "4096x4096"},
        # columns of a table brought to mean 0 and deviation 1: many rows, few features, an odd number of them
        {"name": "standardize 131072x257", "kind": "standardize", "type": "SFloat", "shape": "131072x257"},
        # every other column of a transposed matrix through exp, thresholded and counted; every third row copied
        {"name": "views 8192x8192", "kind": "views", "type": "SFloat", "shape": "8192x8192"},
        # softmax over attention scores, written as a chain of array operations
        {"name": "softmax 32x16x512x512", "kind": "softmax", "type": "SFloat", "shape": "32x16x512x512"},
        # layer normalisation, as a chain and in one call, and softmax in one call, of rows of an odd length
        {"name": "layernorm 8192x4095", "kind": "layernorm", "type": "SFloat", "shape": "8192x4095"},
        # what lies in a range: mask, count, values, positions; and a batch of rows picked by index
        {"name": "select 8192x4096", "kind": "select", "type": "SFloat", "shape": "8192x4096"},
        # running sums of the whole and along either axis in double precision
        {"name": "scan 4096x4096", "kind": "scan", "type": "DFloat", "shape": "4096x4096"},
        # functions of a vector: densities, activations, powers
        {"name": "functions 2^24", "kind": "functions", "type": "SFloat", "shape": "16777216"},
    ]


#: kinds, the types that are drawn for each, and the dimensions (fewest, most)
KINDS = {
    "step": (("SFloat", "SFloat", "DFloat"), 1, 1),
    "reduce": (("SFloat", "SFloat", "DFloat", "Int32"), 2, 3),
    "bias": (("SFloat", "DFloat"), 2, 2),
    "standardize": (("SFloat", "SFloat", "DFloat"), 2, 2),
    "views": (("SFloat", "SFloat", "DFloat"), 2, 2),
    "softmax": (("SFloat", "SFloat", "DFloat"), 2, 4),
    "layernorm": (("SFloat", "SFloat", "DFloat"), 2, 2),
    "select": (("SFloat", "SFloat", "DFloat", "Int32"), 2, 2),
    "scan": (("SFloat", "DFloat"), 2, 2),
    "functions": (("SFloat", "SFloat", "DFloat"), 1, 1),
}


def draw(rng):
    kind = rng.choice(sorted(KINDS))
    types, fewest, most = KINDS[kind]
    kind_type = rng.choice(types)
    # elements: from the shortest vector listed to 2^25, 2^26 for the chain over scores
    n = math.exp(rng.uniform(math.log(10000), math.log(2 ** (26 if kind == "softmax" else 25))))
    dims = []
    for left in range(rng.randint(fewest, most), 1, -1):
        # neither side of a split below 8, the last two dimensions the longer ones
        share = rng.uniform(0.25, 0.75) if left == 2 else rng.uniform(0.1, 0.3)
        d = max(8, int(n ** share))
        dims.append(d)
        n = max(8.0, n / d)
    dims.append(int(n))
    # half of the last dimensions are whole numbers of 16 elements, the other half are what they are
    if rng.random() < 0.5:
        dims[-1] = max(16, dims[-1] // 16 * 16)
    if kind in ("views", "select"):
        # masks come back as whole bytes
        at = 1 if kind == "views" else 0
        dims[at] = max(8, dims[at] // 8 * 8)
    return {"kind": kind, "type": kind_type, "shape": "x".join(str(d) for d in dims)}


def _shape(case):
    return [int(d) for d in case["shape"].split("x")]


# ---------------------------------------------------------------------------
# arrays of the library as tensors on the same memory
# ---------------------------------------------------------------------------
_TYPESTR = {"sfloat": "<f4", "dfloat": "<f8", "int32": "<i4", "int64": "<i8", "uint64": "<i8", "bit": "|u1"}


class _Memory:
    """A contiguous array's memory for torch; holds the array."""

    def __init__(self, a):
        shape = ((a.size + 7) // 8,) if isinstance(a, Bit) else a.shape
        self.array = a
        self.__cuda_array_interface__ = {"shape": shape, "typestr": _TYPESTR[a.type_name], "data": (a._ptr(), False), "version": 2}


def _tensor(a):
    return torch.as_tensor(_Memory(a), device="cuda")


def _filled(cls, shape, fill):
    a = cls(*shape)
    fill(_tensor(a))
    return a


# ---------------------------------------------------------------------------
# what a program has in hand before the pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, cls, shape = case["kind"], CLASS[case["type"]], _shape(case)
    s = {"kind": kind}
    if kind == "step":
        s["x"] = _filled(cls, shape, lambda t: t.uniform_(-1, 1, generator=g))
        s["b"] = _filled(cls, shape, lambda t: t.uniform_(0, 2, generator=g))
    elif kind == "reduce":
        # multiples of 1/16 in [-4, 4), so that ties are met; whole numbers below 1000 for Int32
        def levels(t):
            if cls is Int32:
                t.random_(0, 1000, generator=g)
            else:
                t.random_(-64, 64, generator=g).div_(16)
        s["x"] = _filled(cls, shape, levels)
        s["last"] = len(shape) - 1
        s["float"] = cls is not Int32
    elif kind == "bias":
        s["x"] = _filled(cls, shape, lambda t: t.normal_(0, 1, generator=g))
        s["r"] = _filled(cls, [1, shape[1]], lambda t: t.normal_(1, 1, generator=g))
    elif kind == "standardize":
        # features of different places and scales
        place = torch.empty(shape[1], device="cuda").uniform_(-3, 3, generator=g)
        scale = torch.empty(shape[1], device="cuda").uniform_(0.5, 4, generator=g)
        s["x"] = _filled(cls, shape, lambda t: t.normal_(0, 1, generator=g).mul_(scale).add_(place))
    elif kind == "views":
        s["m"] = _filled(cls, shape, lambda t: t.normal_(0, 1, generator=g))
        s["i"] = _filled(Int32, shape, lambda t: t.random_(0, 1000, generator=g))
    elif kind == "softmax":
        s["x"] = _filled(cls, shape, lambda t: t.normal_(0, 2, generator=g))
    elif kind == "layernorm":
        s["x"] = _filled(cls, shape, lambda t: t.normal_(0.5, 1, generator=g))
    elif kind == "select":
        # the same values in another order for every seed (the quantiles of N(0, 1), or -100 to 99 over and over),
        # so that the selection has one size
        n = shape[0] * shape[1]
        order = torch.randperm(n, generator=g, device="cuda").reshape(shape)
        if cls is Int32:
            s["x"] = _filled(cls, shape, lambda t: t.copy_(order % 200 - 100))
            s["low"], s["high"] = 10, 60
        else:
            s["x"] = _filled(cls, shape, lambda t: t.copy_(torch.special.ndtri((order.double() + 0.5) / n)))
            s["low"], s["high"] = 0.25, 1.5
        s["rows"] = np.random.default_rng(seed).integers(0, shape[0], max(1, shape[0] // 4))
    elif kind == "scan":
        s["x"] = _filled(cls, shape, lambda t: t.uniform_(0, 1, generator=g))
        s["flat"] = s["x"].reshape(s["x"].size)
    elif kind == "functions":
        s["x"] = _filled(cls, shape, lambda t: t.uniform_(0.05, 3, generator=g))
    else:
        raise ValueError(kind)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _step(s):
    y = 2.5 * s["x"] + s["b"]
    c = y - y.mean()
    return [c, y.sum(), c.mulsum(s["b"])]


def _reduce(s):
    x = s["x"]
    got = []
    for axis in list(range(s["last"] + 1)) + [None]:
        got += [x.sum(axis=axis), x.max(axis=axis)]
    got += [x.argmax(axis=s["last"]), x.argmin(axis=0)]
    if s["float"]:
        got += [x.mean(axis=0, keepdims=True), x.var(axis=s["last"])]
    return got


def _bias(s):
    c = s["x"] + s["r"]
    return [c, c.sum(axis=1), c.max(axis=1)]


def _standardize(s):
    x = s["x"]
    m, d = x.mean(axis=0), x.stddev(axis=0)
    low, high = x.minmax(axis=0)
    return [(x - m) / d, m, d, low, high]


def _views(s):
    v = s["m"].transpose()[:, ::2]
    e = NMath.exp(v) - 1.0
    mask = e > 0.5
    return [e, mask, mask.count_true(), s["i"][::3].copy()]


def _softmax(s):
    x = s["x"]
    e = NMath.exp(x - x.max(axis=-1, keepdims=True))
    return [e / e.sum(axis=-1, keepdims=True)]


def _layernorm(s):
    x = s["x"]
    mean, var = x.mean(axis=-1, keepdims=True), x.var(axis=-1, keepdims=True)
    return [(x - mean) / NMath.sqrt(var + 1e-5), mean, var, Fused.layernorm(x, 1e-5), Fused.softmax(x)]


def _select(s):
    x = s["x"]
    mask = (x > s["low"]) & (x < s["high"])
    return [mask, mask.count_true(axis=1), mask.count_true(axis=0), x[mask], mask.where(), x[s["rows"]]]


def _scan(s):
    x = s["x"]
    return [s["flat"].cumsum(), x.cumsum(axis=0), x.cumsum(axis=1)]


def _functions(s):
    x = s["x"]
    return [NMath.log(x), NMath.exp(x), NMath.sin(x), NMath.tanh(x), NMath.erf(x), NMath.erfc(x), NMath.asinh(x), NMath.sqrt(x), x ** 2.7]


PASS = {"step": _step, "reduce": _reduce, "bias": _bias, "standardize": _standardize, "views": _views, "softmax": _softmax,
        "layernorm": _layernorm, "select": _select, "scan": _scan, "functions": _functions}


def run(state):
    return [_tensor(a) for a in PASS[state["kind"]](state)]


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind, shape, w = case["kind"], _shape(case), SIZE[case["type"]]
    n, last = math.prod(shape), shape[-1]
    rows = n // last
    b = w * n                            # one read or one write of the array
    if kind == "step":
        # 2.5 * x, + b, mean, - mean, sum, mulsum
        return {"bytes": (2 + 3 + 1 + 2 + 1 + 2) * b, "flops": 7 * n}
    if kind == "reduce":
        out = sum(2 * w * n // d for d in shape) + 4 * rows + 4 * n // shape[0]
        calls = 2 * (len(shape) + 1) + 2
        if case["type"] != "Int32":
            calls += 2
            out += w * n // shape[0] + w * rows
        return {"bytes": calls * b + out, "flops": (calls + 2) * n}
    if kind == "bias":
        return {"bytes": 4 * b + w * last + 2 * w * rows, "flops": 3 * n}
    if kind == "standardize":
        # mean, stddev, minmax, - m, / d
        return {"bytes": 7 * b + 6 * w * last, "flops": 8 * n}
    if kind == "views":
        v = shape[1] * ((shape[0] + 1) // 2)
        i = 4 * shape[1] * ((shape[0] + 2) // 3)
        return {"bytes": 5 * w * v + 2 * v // 8 + 2 * i, "flops": 3 * v}
    if kind == "softmax":
        # max, - max, exp, sum, / sum
        return {"bytes": 8 * b + 4 * w * rows, "flops": 5 * n}
    if kind == "layernorm":
        # mean, var, - mean, / sqrt(var + eps); the two calls
        return {"bytes": 10 * b + 8 * w * rows, "flops": 18 * n}
    if kind == "select":
        hit = 0.332 if case["type"] != "Int32" else 0.245
        # two comparisons, and; counts along rows and columns, where, mask, and its positions; the values; the batch
        bits = (2 + 3 + 2 + 2) * n // 8
        batch = max(1, shape[0] // 4)
        return {"bytes": 2 * b + bits + int((4 + 2 * w) * hit * n) + 2 * w * batch * last + 8 * (rows + last + batch), "flops": 4 * n}
    if kind == "scan":
        return {"bytes": 6 * b, "flops": 3 * n}
    return {"bytes": 18 * b, "flops": 9 * n}


def tolerance(case):
    # Against the same pass in 64 bits, DFloat against sums in another order: SFloat is off by up to 2.3e-7 in norm (a
    # dot product of a centred vector) and 2.3e-6 in one value (a column whose deviation is small against its mean),
    # DFloat by 2.2e-15 and 1.0e-14 (running sums of 3e7 elements); about four times that. Positions, masks, counts
    # and whatever holds whole numbers are the same.
    if case["type"] == "Int32":
        return "exact"
    return {"rel": 1e-6, "max": 1e-5} if case["type"] == "SFloat" else {"rel": 1e-14, "max": 4e-14}
