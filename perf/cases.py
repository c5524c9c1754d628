"""What a program on this backend spends its time in: twelve workloads over the public entry points.

Each case runs one pass through `nx_amd.nx` (eager), `nx_amd.defn` (traced once, called many times) or
`nx_amd.random`, on tensors that are on the device already.  `listed()` are the fixed ones, `draw(rng)` gives
further sizes, types and layouts of the same workloads.  Inputs are made on the device with torch and handed to
the backend by pointer; results stay device tensors and are looked at through torch views.
"""
from __future__ import annotations

import math

import torch

from nx_amd import defn
from nx_amd import nx as Nx
from nx_amd import random as Random
from nx_amd.backend import HipNxBackend
from nx_amd.tensor import Tensor

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "s8": torch.int8}
_BYTES = {"f32": 4, "bf16": 2, "f16": 2, "s8": 1}


# ---- tensors in, tensors out ----------------------------------------------------------------------

def _nx(t: torch.Tensor) -> Tensor:
    """A dense torch tensor on the device as a tensor of the backend, over the same memory."""
    t = t.contiguous()
    name = next(n for n, d in _TORCH.items() if d == t.dtype)
    pointer = Nx.Pointer(kind="local", address=t.data_ptr(), data_size=t.numel() * t.element_size())
    return Nx.from_pointer(HipNxBackend, pointer, name, tuple(t.shape), keep=t)


class _Memory:
    """The device memory of a backend tensor, as torch takes it over; holds the tensor."""

    def __init__(self, t: Tensor, code: str):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": code, "version": 2,
                                         "data": (Nx.to_pointer(t).address, False)}


def _torch(t: Tensor) -> torch.Tensor:
    kind, bits = t.type
    code = "<%s%d" % ("f" if kind == "f" else "i", bits // 8)  # (bf16 as its bits; u32 positions stay below 2^31)
    view = torch.as_tensor(_Memory(t, code), device="cuda")
    return view.view(torch.bfloat16) if kind == "bf" else view


class Results(tuple):
    """The device tensors of one pass, as a program holds them; going through them gives torch views."""

    def __iter__(self):
        return (_torch(t) for t in tuple.__iter__(self))


# ---- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # a small eager chain, sum(exp((a + b) * 0.5)) along rows: four callbacks whose launches are what counts
        {"name": "chain_f32_1024", "kind": "chain", "rows": 1024, "cols": 1024, "type": "f32"},
        # feature standardisation of a table along its first axis, eager: column sums and broadcasts over 268 MB
        {"name": "standardise_f32_671088x100", "kind": "standardise", "rows": 671088, "cols": 100, "type": "f32"},
        # probabilities over a vocabulary, traced with compiled groups
        {"name": "softmax_f32_8192x32000", "kind": "softmax", "rows": 8192, "cols": 32000, "type": "f32"},
        # layer normalisation with gain and bias, traced with compiled groups
        {"name": "layer_norm_f32_16384x1024", "kind": "layer_norm", "rows": 16384, "cols": 1024, "type": "f32"},
        # attention probabilities of a prompt from projected activations: heads split off, scores, scaling, softmax
        {"name": "attention_bf16_4x8x512x64", "kind": "attention", "batch": 4, "heads": 8, "queries": 512, "keys": 512,
         "dim": 64, "type": "bf16"},
        # the large square contraction
        {"name": "dot_bf16_4096", "kind": "dot", "m": 4096, "n": 4096, "k": 4096, "type": "bf16", "weights": "k_outer"},
        # a contraction of ordinary size none of whose extents is a power of two
        {"name": "dot_bf16_2000x3000x1000", "kind": "dot", "m": 2000, "n": 3000, "k": 1000, "type": "bf16", "weights": "k_outer"},
        # an int8 weight-only linear layer over a serving batch, scales per output column
        {"name": "int8_linear_64x11008x4096", "kind": "int8_linear", "m": 64, "n": 11008, "k": 4096, "weights": "k_inner"},
        # the same layer in bf16 while a few sequences are decoded: a stream of the weights
        {"name": "linear_bf16_8x11008x4096", "kind": "dot", "m": 8, "n": 11008, "k": 4096, "type": "bf16", "weights": "k_outer"},
        # one training step of a two-layer classifier in f32: forward, backward, update
        {"name": "train_f32_4096x784x512x10", "kind": "train", "batch": 4096, "inputs": 784, "hidden": 512, "classes": 10},
        # greedy choice over a vocabulary and the rows of the embedding table it picks
        {"name": "argmax_take_8192x32000", "kind": "pick", "rows": 8192, "vocab": 32000, "width": 4096},
        # normally distributed f32 samples from a key (initial weights, noise), traced with compiled groups
        {"name": "normal_f32_2p26", "kind": "normal", "count": 1 << 26},
    ]


def _log(rng, low, high, odd=0.5):
    """A size between `low` and `high`, spread over its logarithm; half of them as they fall, half in eights."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return max(low, min(high, n if rng.random() < odd else max(8, n // 8 * 8)))


def draw(rng):
    kind = rng.choice(["chain", "standardise", "softmax", "layer_norm", "attention", "dot", "dot", "int8_linear", "train",
                       "pick", "normal"])
    if kind in ("chain", "standardise", "softmax", "layer_norm"):
        cols = {"chain": lambda: _log(rng, 16, 16384), "standardise": lambda: _log(rng, 2, 2048),
                "softmax": lambda: _log(rng, 64, 32000), "layer_norm": lambda: _log(rng, 64, 8192)}[kind]()
        rows = _log(rng, 16, max(16, min(1 << 20, (1 << 26) // cols)))
        return {"kind": kind, "rows": rows, "cols": cols, "type": rng.choice(["f32", "f32", "bf16"])}
    if kind == "attention":
        batch, heads, dim = _log(rng, 1, 8, 1), rng.choice([4, 8, 12, 16]), rng.choice([64, 128])
        keys = _log(rng, 64, 2048)
        queries = 1 if rng.random() < 0.3 else _log(rng, 64, 1024)  # one: a step of decoding
        while batch * heads * queries * keys > 1 << 26:
            queries = max(1, queries // 2)
        return {"kind": kind, "batch": batch, "heads": heads, "queries": queries, "keys": keys, "dim": dim,
                "type": rng.choice(["bf16", "f16"])}
    if kind == "dot":
        weights = rng.choice(["k_outer", "k_inner"])
        if rng.random() < 0.4:  # the rows of a serving batch against a long matrix
            return {"kind": kind, "m": _log(rng, 1, 128), "n": _log(rng, 128, 11008), "k": _log(rng, 128, 11008),
                    "type": rng.choice(["bf16", "bf16", "f16"]), "weights": weights}
        ty = rng.choice(["bf16", "bf16", "f16", "f32"])
        m, n, k = (_log(rng, 128, 2048 if ty == "f32" else 4096) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k, "type": ty, "weights": weights}
    if kind == "int8_linear":
        return {"kind": kind, "m": _log(rng, 1, 512), "n": _log(rng, 256, 11008), "k": _log(rng, 256, 11008),
                "weights": rng.choice(["k_inner", "k_outer"])}
    if kind == "train":
        return {"kind": kind, "batch": _log(rng, 32, 8192), "inputs": _log(rng, 64, 1024), "hidden": _log(rng, 64, 1024),
                "classes": _log(rng, 2, 100)}
    if kind == "pick":
        vocab = _log(rng, 1000, 50257)
        return {"kind": kind, "rows": _log(rng, 1, min(8192, (1 << 28) // vocab)), "vocab": vocab, "width": _log(rng, 64, 4096)}
    return {"kind": "normal", "count": _log(rng, 1 << 12, 1 << 26)}


# ---- what a program writes ------------------------------------------------------------------------

def _chain(a, b):
    return Nx.sum(Nx.exp(Nx.multiply(Nx.add(a, b), 0.5)), axes=[1])


def _standardise(x):
    mean = Nx.mean(x, axes=[0], keep_axes=True)
    centred = Nx.subtract(x, mean)
    variance = Nx.mean(Nx.multiply(centred, centred), axes=[0], keep_axes=True)
    return Nx.multiply(centred, Nx.rsqrt(Nx.add(variance, 1.0e-5))), mean, variance


def _softmax(x):
    e = Nx.exp(Nx.subtract(x, Nx.reduce_max(x, axes=[-1], keep_axes=True)))
    return Nx.divide(e, Nx.sum(e, axes=[-1], keep_axes=True))


def _layer_norm(x, gain, bias):
    mean = Nx.mean(x, axes=[-1], keep_axes=True)
    centred = Nx.subtract(x, mean)
    variance = Nx.mean(Nx.multiply(centred, centred), axes=[-1], keep_axes=True)
    return Nx.add(Nx.multiply(Nx.multiply(centred, Nx.rsqrt(Nx.add(variance, 1.0e-5))), gain), bias)


def _attention(heads, dim):
    def probabilities(q, k):
        q = Nx.transpose(Nx.reshape(q, (q.shape[0], q.shape[1], heads, dim)), axes=[0, 2, 1, 3])
        k = Nx.transpose(Nx.reshape(k, (k.shape[0], k.shape[1], heads, dim)), axes=[0, 2, 1, 3])
        scores = Nx.dot(q, [3], [0, 1], k, [3], [0, 1])
        return _softmax(Nx.multiply(Nx.as_type(scores, "f32"), 1.0 / math.sqrt(dim)))
    return probabilities


def _int8_linear(contract):
    def layer(x, w, scales):
        return Nx.multiply(Nx.as_type(Nx.dot(x, [1], w, [contract], out_type="s32"), "f32"), scales)
    return layer


def _train(x, y, w1, b1, w2, b2):
    """Softmax cross-entropy of relu(x w1 + b1) w2 + b2 against one-hot rows `y`; one step of gradient descent."""
    pre = Nx.add(Nx.dot(x, w1), b1)
    hidden = Nx.max(pre, 0.0)
    probabilities = _softmax(Nx.add(Nx.dot(hidden, w2), b2))
    loss = Nx.divide(Nx.sum(Nx.multiply(y, Nx.log(Nx.add(probabilities, 1.0e-7)))), -x.shape[0])
    d_logits = Nx.divide(Nx.subtract(probabilities, y), x.shape[0])
    d_w2 = Nx.dot(hidden, [0], d_logits, [0])
    d_pre = Nx.multiply(Nx.dot(d_logits, [1], w2, [1]), Nx.greater(pre, 0.0))
    d_w1 = Nx.dot(x, [0], d_pre, [0])

    def step(value, gradient):
        return Nx.subtract(value, Nx.multiply(gradient, 0.1))
    return (loss, step(w1, d_w1), step(b1, Nx.sum(d_pre, axes=[0])), step(w2, d_w2), step(b2, Nx.sum(d_logits, axes=[0])))


def prepare(case, seed):
    Nx.default_backend(HipNxBackend, {"device": 0})
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = case["kind"]
    dtype = _TORCH[case.get("type", "f32")]

    def normal(*shape, scale=1.0, dtype=dtype):
        t = torch.empty(shape, device="cuda", dtype=torch.float32).normal_(0.0, scale, generator=g)
        return t.to(dtype)

    def uniform(*shape, low, high, dtype=dtype):
        return torch.empty(shape, device="cuda", dtype=torch.float32).uniform_(low, high, generator=g).to(dtype)

    def whole(*shape):
        return torch.randint(-127, 128, shape, device="cuda", dtype=torch.int8, generator=g)

    if kind == "chain":
        args, fun = [uniform(case["rows"], case["cols"], low=-1, high=1) for _ in range(2)], _chain
    elif kind == "standardise":
        args, fun = [normal(case["rows"], case["cols"], scale=2.0) + 1], _standardise
    elif kind == "softmax":
        args, fun = [normal(case["rows"], case["cols"], scale=2.0)], _softmax
    elif kind == "layer_norm":
        cols = case["cols"]
        args, fun = [normal(case["rows"], cols), uniform(cols, low=0.5, high=1.5), normal(cols, scale=0.1)], _layer_norm
    elif kind == "attention":
        width = case["heads"] * case["dim"]
        args = [normal(case["batch"], case["queries"], width), normal(case["batch"], case["keys"], width)]
        fun = _attention(case["heads"], case["dim"])
    elif kind in ("dot", "int8_linear"):
        k_inner = case["weights"] == "k_inner"
        m, k, right = case["m"], case["k"], (case["n"], case["k"]) if k_inner else (case["k"], case["n"])
        if kind == "dot":
            args = [normal(m, k, scale=1 / 64), normal(*right, scale=1 / 64)]
            fun = lambda x, w: Nx.dot(x, [1], w, [1 if k_inner else 0])  # noqa: E731
        else:
            args = [whole(m, k), whole(*right), uniform(case["n"], low=1e-3, high=1e-2)]
            fun = _int8_linear(1 if k_inner else 0)
    elif kind == "train":
        batch, inputs, hidden, classes = (case[n] for n in ("batch", "inputs", "hidden", "classes"))
        labels = torch.randint(0, classes, (batch,), device="cuda", generator=g)
        args = [uniform(batch, inputs, low=0, high=1), torch.nn.functional.one_hot(labels, classes).to(torch.float32),
                normal(inputs, hidden, scale=inputs ** -0.5), normal(hidden, scale=0.01),
                normal(hidden, classes, scale=hidden ** -0.5), normal(classes, scale=0.01)]
        fun = _train
    elif kind == "pick":
        logits = normal(case["rows"], case["vocab"], scale=2.0)
        tied = torch.randperm(case["rows"], device="cuda", generator=g)[: max(case["rows"] // 100, 1)]  # ties of the maximum
        at = torch.randint(0, case["vocab"], (len(tied),), device="cuda", generator=g)
        logits[tied, at] = logits[tied].amax(dim=1)
        args = [logits, normal(case["vocab"], case["width"], scale=0.02, dtype=torch.bfloat16)]

        def fun(logits, table):
            best = Nx.argmax(logits, axis=1, type="u32")
            return best, Nx.take(table, best)
    else:
        args = []
        key, count = Random.key(seed, backend=HipNxBackend), case["count"]

        def fun(key):
            return Random.normal(key, shape=(count,))
    args = [_nx(a) for a in args] if args else [key]
    if kind in ("softmax", "layer_norm", "attention", "int8_linear", "train", "normal"):
        fun = defn.compile(fun, *args, fuse="compiled")
    torch.cuda.synchronize()  # the inputs are there before the backend's own stream reads them
    return {"fun": fun, "args": args}


def run(state):
    out = state["fun"](*state["args"])
    return Results(out if isinstance(out, (tuple, list)) else (out,))


def work(case):
    kind = case["kind"]
    size = _BYTES[case.get("type", "f32")]
    if kind in ("chain", "standardise", "softmax", "layer_norm"):
        n, cols = case["rows"] * case["cols"], case["cols"]
        moved = {"chain": 2 * n + case["rows"], "standardise": 2 * n + 2 * cols, "softmax": 2 * n, "layer_norm": 2 * n + 2 * cols}[kind]
        return {"bytes": moved * size, "flops": {"chain": 4, "standardise": 7, "softmax": 5, "layer_norm": 9}[kind] * n}
    if kind == "attention":
        rows, width = case["batch"] * case["heads"] * case["queries"], case["heads"] * case["dim"]
        return {"bytes": case["batch"] * (case["queries"] + case["keys"]) * width * size + 4 * rows * case["keys"],
                "flops": rows * case["keys"] * (2 * case["dim"] + 6)}
    if kind in ("dot", "int8_linear"):
        m, n, k = case["m"], case["n"], case["k"]
        if kind == "dot":
            return {"bytes": (m * k + k * n + m * n) * size, "flops": 2 * m * n * k}
        return {"bytes": m * k + k * n + 4 * (m * n + n), "flops": 2 * m * n * k}
    if kind == "train":
        b, i, h, c = (case[n] for n in ("batch", "inputs", "hidden", "classes"))
        return {"bytes": 4 * (b * (i + c) + 2 * (i * h + h + h * c + c)), "flops": 4 * b * i * h + 6 * b * h * c}
    if kind == "pick":
        rows = case["rows"]
        return {"bytes": 4 * rows * case["vocab"] + 4 * rows + 4 * rows * case["width"], "flops": 0}
    return {"bytes": 4 * case["count"], "flops": 0}


# About four times how far each workload lies from itself in 64 bits (relative 2-norm, largest difference), over the
# listed cases and drawn ones: the rounding of its own types, bf16 results dropping their low bits as the backend does.
_TOLERANCE = {
    ("chain", "f32"): (1.5e-7, 3.0e-7), ("chain", "bf16"): (2.8e-2, 4.0e-2),
    ("standardise", "f32"): (2.5e-7, 1.0e-6), ("standardise", "bf16"): (3.0e-2, 1.2e-1),
    ("softmax", "f32"): (3.5e-7, 2.0e-6), ("softmax", "bf16"): (3.0e-2, 1.2e-1),
    ("layer_norm", "f32"): (3.0e-7, 1.5e-6), ("layer_norm", "bf16"): (3.0e-2, 1.2e-1),
    ("attention", "bf16"): (2.4e-2, 1.0e-1), ("attention", "f16"): (2.0e-3, 8.0e-3),
    ("dot", "bf16"): (1.3e-2, 3.2e-2), ("dot", "f16"): (1.0e-3, 2.0e-3), ("dot", "f32"): (4.0e-6, 3.0e-5),
    ("train", "f32"): (3.5e-7, 1.5e-6), ("normal", "f32"): (3.2e-7, 9.0e-7),
}


def tolerance(case):
    if case["kind"] in ("pick", "int8_linear"):  # positions and copied rows; whole sums, and one rounded product of each
        return "exact"
    rel, largest = _TOLERANCE[case["kind"], case.get("type", "f32")]
    return {"rel": rel, "max": largest}
