"""The work whose speed this library answers for, through its public entry points.

Four kinds of pass:

* ``mul``: one ``marlin.mul`` into a C that the caller keeps -- fp16 rows times
  4-bit weights in Marlin format.
* ``layers``: one forward pass through the quantised linear layers of a stack
  of blocks (``marlin.Layer``), as a decoder calls them, each layer with
  weights and activations of its own.
* ``dense``: one ``streamk.gemm``, fp16 times fp16, C allocated by the call.
* ``convert``: a layer's fp16 weight quantised and packed
  (``marlin.quantize``, ``marlin.Layer.pack``), what loading a model costs per
  layer.

Values are distributed as in the tests and the benchmark: activations N(0, 1),
4-bit weights uniform, scales U(0.001, 0.02), dense operands U(-2, 2), weights
to be quantised N(0, 0.02).
"""
import os
import sys

import torch

# the package's folder is no identifier: its modules are imported by themselves
sys.path.insert(0, os.path.join(os.path.abspath(os.getcwd()), "awesome-cute_amd"))
import marlin  # noqa: E402
import streamk  # noqa: E402

DEV = "cuda:0"


def _mul(m, n, k, group, name=None):
    return _named(name, kind="mul", m=m, n=n, k=k, group=group)


def _layers(m, shapes, blocks, group, name=None):
    return _named(name, kind="layers", m=m, shapes=shapes, blocks=blocks, group=group)


def _dense(m, n, k, name=None):
    return _named(name, kind="dense", m=m, n=n, k=k)


def _convert(n, k, group, name=None):
    return _named(name, kind="convert", n=n, k=k, group=group)


def _named(name, **case):
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest product of the tests, as a layer: what a call costs by itself
        _layers(16, "256x512", 1, 128, "smallest"),
        # one token, one square layer (attention output of a 7B model): the
        # call that a decoder makes most often
        _mul(1, 4096, 4096, 128, "decode"),
        # one token through the linear layers of four 7B blocks (qkv, attention
        # output, gate and up, down), every weight read from memory
        _layers(1, "12288x4096 4096x4096 21504x4096 4096x10752", 4, 128, "decode_blocks"),
        # sixteen sequences decoded together through the up and down projections
        # of an MLP
        _layers(16, "11008x4096 4096x11008", 1, 128, "batch16_mlp"),
        # a full decoding batch over the largest layer, scales per group ...
        _mul(64, 28672, 8192, 128, "batch64_large"),
        # ... and an uneven batch (speculative decoding, continuous batching)
        # over a qkv projection with one scale per column
        _mul(45, 12288, 4096, -1, "batch45_per_channel"),
        # a short prompt, or a chunk of one beside running decodes: a row count
        # no tile divides over the down projection of a 13B model
        _mul(203, 5120, 13568, 128, "chunk203"),
        # a prompt of 2048 tokens
        _mul(2048, 4096, 4096, 128, "prefill2048"),
        # the largest: a batch of long prompts over the largest layer
        _mul(8192, 28672, 8192, 128, "prefill8192_large"),
        # the dense GEMM on the size its program runs by default (one whole
        # wave of tiles and a partial one)
        _dense(4096, 4352, 4096, "dense"),
        # few and odd rows against deep weights
        _dense(777, 4352, 10240, "dense_ragged"),
        # loading a model: one layer of it
        _convert(11008, 4096, 128, "convert"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _step(rng, lo, hi, step):
    return max(lo, min(hi, step * round(_log(rng, lo, hi) / step)))


def draw(rng):
    kind = rng.choice(["few", "few", "layers", "batch", "batch", "prefill", "prefill", "dense", "dense",
                       "convert"])
    group = rng.choice([128, 128, -1])
    if kind == "few":  # decoding, one to sixteen sequences
        return _mul(_log(rng, 1, 16), _step(rng, 256, 28672, 256), _step(rng, 512, 21760, 128), group)
    if kind == "layers":
        hidden = _step(rng, 1024, 8192, 256)
        inner = _step(rng, hidden, 3 * hidden, 256)
        shapes = f"{3 * hidden}x{hidden} {hidden}x{hidden} {2 * inner}x{hidden} {hidden}x{inner}"
        return _layers(_log(rng, 1, 16), shapes, rng.choice([1, 2]), group)
    if kind == "batch":  # larger batches and chunks of prompts
        return _mul(_log(rng, 17, 320), _step(rng, 512, 28672, 256), _step(rng, 1024, 13824, 128), group)
    if kind == "prefill":
        return _mul(_log(rng, 321, 8192), _step(rng, 1024, 28672, 256), _step(rng, 1024, 8192, 128), group)
    if kind == "dense":
        return _dense(_log(rng, 64, 8192), _step(rng, 512, 8192, 256), _step(rng, 512, 10240, 64))
    return _convert(_step(rng, 1024, 28672, 256), _step(rng, 1024, 8192, 128), group)


def _quantised(n, k, group, gen):
    B = torch.randint(-2 ** 31, 2 ** 31, (k // 16, 2 * n), dtype=torch.int32, device=DEV, generator=gen)
    rows = 1 if group == -1 else k // group
    s = (torch.rand((rows, n), device=DEV, generator=gen) * 0.019 + 0.001).half()
    return B, s


def _shapes(case):
    return [tuple(int(x) for x in s.split("x")) for s in case["shapes"].split()] * case["blocks"]


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, dtype=torch.half, device=DEV, generator=gen)

    state = {"kind": case["kind"]}
    if case["kind"] == "mul":
        m, n, k = case["m"], case["n"], case["k"]
        state["B"], state["s"] = _quantised(n, k, case["group"], gen)
        state["A"] = randn(m, k)
        state["C"] = torch.empty((m, n), dtype=torch.half, device=DEV)
        state["workspace"] = torch.zeros(n // 128 * 16, dtype=torch.int32, device=DEV)
    elif case["kind"] == "layers":
        state["layers"] = []
        for n, k in _shapes(case):
            with torch.device(DEV):
                layer = marlin.Layer(k, n, case["group"])
            layer.B, layer.s = _quantised(n, k, case["group"], gen)
            state["layers"].append((layer, randn(case["m"], k)))
    elif case["kind"] == "dense":
        m, n, k = case["m"], case["n"], case["k"]
        state["A"] = (torch.rand((m, k), device=DEV, generator=gen) * 4 - 2).half()
        state["B"] = (torch.rand((n, k), device=DEV, generator=gen) * 4 - 2).half()
    else:
        n, k = case["n"], case["k"]
        with torch.device(DEV):
            state["linear"] = torch.nn.Linear(k, n, bias=False, dtype=torch.half)
            state["layer"] = marlin.Layer(k, n, case["group"])
        state["w"] = randn(k, n) * 0.02
        state["group"] = case["group"]
    return state


def run(state):
    if state["kind"] == "mul":
        marlin.mul(state["A"], state["B"], state["C"], state["s"], state["workspace"])
        return state["C"]
    if state["kind"] == "layers":
        return [layer(x) for layer, x in state["layers"]]
    if state["kind"] == "dense":
        return streamk.gemm(state["A"], state["B"])
    fake, q, s = marlin.quantize(state["w"], state["group"])
    state["linear"].weight.data = fake.t()
    state["layer"].pack(state["linear"], s.t())
    return {"weight": fake, "q": q, "scales": s, "B": state["layer"].B, "s": state["layer"].s}


def work(case):
    def product(m, n, k):
        groups = 1 if case["group"] == -1 else k // case["group"]
        return n * k / 2 + 2 * groups * n + 2 * m * (n + k), 2 * m * n * k

    if case["kind"] == "mul":
        b, f = product(case["m"], case["n"], case["k"])
    elif case["kind"] == "layers":
        each = [product(case["m"], n, k) for n, k in _shapes(case)]
        b, f = sum(x[0] for x in each), sum(x[1] for x in each)
    elif case["kind"] == "dense":
        m, n, k = case["m"], case["n"], case["k"]
        b, f = 2 * (m * k + n * k + m * n), 2 * m * n * k
    else:
        n, k = case["n"], case["k"]
        groups = 1 if case["group"] == -1 else k // case["group"]
        # w read; fake weight, q (32 bits), scales, packed words and scales written
        b, f = n * k * (2 + 2 + 4 + 0.5) + 4 * groups * n, 4 * n * k
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # whole numbers, and halves that one defined sequence of roundings gives
    if case["kind"] == "convert":
        return "exact"
    # four times what the kernels showed against float64 products of the exact
    # operands: the rounding of the result (2.1e-4), and with 4-bit weights that
    # of the weights or the scaled sums (2.7e-4 to 3.0e-4, worst element 1.1e-3)
    if case["kind"] == "dense":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 1.2e-3, "max": 5e-3}
