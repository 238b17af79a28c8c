"""The work that programs of this framework have it do, as measurable cases.

A case is one tile program of ``xtile_amd.kernels`` at one size, planned once
(``xt.compile``) and launched over device tensors that the caller owns
(``xt.launch``), as a program that serves or trains with these kernels calls
them.  ``listed`` holds fixed cases from the smallest calls to the largest,
``draw`` gives more from the same ranges.
"""

from __future__ import annotations

import math

import torch

import xtile_amd as xt
from xtile_amd import kernels as K

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8}
_DSL = {"f16": xt.float16, "bf16": xt.bfloat16, "i8": xt.int8}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1}

# No drawn case costs more than the largest listed ones.
_MAX_ELEMENTS = 8192 * 4096
_MAX_FLOPS = 2 * 4096 * 11008 * 4096


def listed():
    return [
        # A call on a small array, where what counts is the launch: glue
        # between larger kernels, short vectors, single tokens.
        {"name": "add_small", "kind": "add", "rows": 64, "cols": 128, "trow": 32, "tcol": 64},
        # A residual sum over a whole activation array, the reference's
        # full-width row tiles: far beyond the caches.
        {"name": "add_rows_large", "kind": "add_rows", "rows": 8192, "cols": 4096, "trow": 64},
        # The row softmax configuration of the benchmark: one row a Block.
        {"name": "softmax_wide", "kind": "softmax", "rows": 8192, "cols": 4096, "trow": 1},
        # Class scores: a row length that is no power of two, several rows a
        # Block as in the reference's softmax program.
        {"name": "softmax_classes", "kind": "softmax", "rows": 5000, "cols": 1000, "trow": 8},
        # Layer normalisation of a middle-sized model's activations.
        {"name": "layernorm_768", "kind": "layernorm", "rows": 4096, "cols": 768, "trow": 4},
        # An ordinary dense layer.
        {"name": "matmul_f16_1024", "kind": "matmul", "dtype": "f16", "m": 1024, "n": 1024, "k": 1024, "tm": 128,
         "tn": 128},
        # The benchmark's rectangular product: a feed-forward layer of a large
        # model over many tokens.
        {"name": "matmul_bf16_large", "kind": "matmul", "dtype": "bf16", "m": 4096, "n": 11008, "k": 4096, "tm": 256,
         "tn": 128},
        # Sizes that no tile of 64 divides: 40 x 40 is the largest square tile
        # that divides 1000 and whose panels fit on chip.
        {"name": "matmul_f16_ragged", "kind": "matmul", "dtype": "f16", "m": 1000, "n": 1000, "k": 1000, "tm": 40,
         "tn": 40},
        # Decoding with 8-bit weights: a few dozen tokens through one layer,
        # the reference's matmul program with its scale / bias / int8 epilogue.
        {"name": "matmul_i8_decode", "kind": "matmul", "dtype": "i8", "m": 64, "n": 4096, "k": 4096, "tm": 64,
         "tn": 64},
        # A middle layer of an image network.
        {"name": "conv_f16_28", "kind": "conv", "dtype": "f16", "n": 32, "h": 28, "w": 28, "cin": 128, "cout": 128,
         "kh": 3, "kw": 3, "stride": 1, "th": 4, "tw": 28},
        # A downsampling layer of the same network in the reference's own type.
        {"name": "conv_i8_down", "kind": "conv", "dtype": "i8", "n": 32, "h": 56, "w": 56, "cin": 64, "cout": 128,
         "kh": 3, "kw": 3, "stride": 2, "th": 4, "tw": 28},
        # Attention of many heads over a window of keys, a tile of queries a
        # Block.
        {"name": "attention_256", "kind": "attention", "dtype": "f16", "heads": 64, "nq": 512, "nk": 256, "d": 64,
         "tq": 64},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _divisor(rng, n, most):
    return rng.choice([d for d in range(1, min(n, most) + 1) if n % d == 0])


def _draw_add(rng):
    while True:
        trow, tcol = _log(rng, 8, 64), _log(rng, 16, 256)
        rows, cols = trow * _log(rng, 1, 512), tcol * _log(rng, 1, 256)
        if 64 * 128 <= rows * cols <= _MAX_ELEMENTS:
            return {"kind": "add", "rows": rows, "cols": cols, "trow": trow, "tcol": tcol}


def _draw_softmax(rng):
    while True:
        trow, cols = rng.choice((1, 2, 4, 8)), _log(rng, 64, 8192)
        if cols > 2048:
            cols -= cols % 4  # longer rows are held as vectors of four
        rows = trow * _log(rng, 16, 8192)
        if rows * cols <= _MAX_ELEMENTS:
            return {"kind": "softmax", "rows": rows, "cols": cols, "trow": trow}


def _draw_layernorm(rng):
    while True:
        cols = _log(rng, 64, 8192)
        trow = rng.choice((1, 2, 4)) if cols <= 1024 else 1
        rows = trow * _log(rng, 16, 8192)
        if rows * cols <= _MAX_ELEMENTS:
            return {"kind": "layernorm", "rows": rows, "cols": cols, "trow": trow}


def _draw_matmul(rng):
    dtype = rng.choice(("f16", "bf16", "i8"))
    while True:
        if dtype != "i8" and rng.random() < 0.3:  # sizes that 64 does not divide
            tm, tn, k = rng.randint(16, 48), rng.randint(16, 48), _log(rng, 64, 1024)
            m, n = tm * _log(rng, 1, 64), tn * _log(rng, 1, 64)
            if (tm + tn) * k * 2 > 150 * 1024:
                continue
        else:
            tm, tn = rng.choice((64, 128)), rng.choice((64, 128))
            m, n, k = tm * _log(rng, 1, 64), tn * _log(rng, 4, 86), 128 * rng.randint(2, 64)
        if 2 * m * n * k <= _MAX_FLOPS:
            return {"kind": "matmul", "dtype": dtype, "m": m, "n": n, "k": k, "tm": tm, "tn": tn}


def _draw_conv(rng):
    while True:
        dtype = rng.choice(("f16", "bf16", "i8"))
        n, size = _log(rng, 1, 64), _log(rng, 7, 112)
        cin = rng.choice((3, 16, 32, 40, 64, 96, 128, 256, 512))
        cout = rng.choice((16, 32, 64, 96, 128, 256, 512))
        kernel = rng.choice((1, 3, 3, 5, 7) if cin <= 64 else (1, 3, 3))
        stride = rng.choice((1, 1, 2))
        out = (size + 2 * (kernel // 2) - kernel) // stride + 1
        flops = 2 * n * out * out * cout * kernel * kernel * cin
        if flops <= _MAX_FLOPS // 8 and n * size * size * cin <= _MAX_ELEMENTS and n * out * out * cout <= _MAX_ELEMENTS:
            return {"kind": "conv", "dtype": dtype, "n": n, "h": size, "w": size, "cin": cin, "cout": cout,
                    "kh": kernel, "kw": kernel, "stride": stride, "th": _divisor(rng, out, 8), "tw": out}


def _draw_attention(rng):
    while True:
        dtype = rng.choice(("f16", "bf16"))
        d, tq, nk = rng.choice((32, 64, 128)), rng.choice((16, 32, 64)), 8 * rng.randint(4, 32)
        heads, nq = _log(rng, 8, 256), tq * _log(rng, 1, 16)
        if nk * d * 6 + tq * (nk + d) * 4 <= 140 * 1024:
            return {"kind": "attention", "dtype": dtype, "heads": heads, "nq": nq, "nk": nk, "d": d, "tq": tq}


def draw(rng):
    return rng.choice((_draw_add, _draw_softmax, _draw_layernorm, _draw_matmul, _draw_matmul, _draw_conv, _draw_conv,
                       _draw_attention))(rng)


def _out_hw(case):
    pad = case["kh"] // 2, case["kw"] // 2
    return ((case["h"] + 2 * pad[0] - case["kh"]) // case["stride"] + 1,
            (case["w"] + 2 * pad[1] - case["kw"]) // case["stride"] + 1)


def _module(case):
    """The case's tile program, traced and parsed."""
    c = case
    if c["kind"] == "add":
        return K.add(c["rows"], c["cols"], c["trow"], c["tcol"])
    if c["kind"] == "add_rows":
        return K.add_rows(c["rows"], c["cols"], c["trow"])
    if c["kind"] == "softmax":
        return K.softmax(c["rows"], c["cols"], c["trow"])
    if c["kind"] == "layernorm":
        return K.layernorm(c["rows"], c["cols"], c["trow"])
    if c["kind"] == "matmul":
        build = {"f16": K.matmul_f16, "bf16": K.matmul_bf16, "i8": K.matmul_i8}[c["dtype"]]
        return build(c["m"], c["n"], c["k"], c["tm"], c["tn"])
    if c["kind"] == "conv":
        return K.conv2d(c["n"], c["h"], c["w"], c["cin"], c["cout"], c["kh"], c["kw"], c["th"], c["tw"],
                        dtype=_DSL[c["dtype"]], stride=(c["stride"], c["stride"]))
    return K.attention(c["heads"], c["nq"], c["nk"], c["d"], c["tq"], qk=_DSL[c["dtype"]])


def _inputs(case, seed):
    """The case's input tensors by name, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0, dtype="f32"):
        return (torch.randn(*shape, generator=g, device="cuda") * std).to(_TORCH[dtype])

    def uniform(*shape, lo=-1.0, hi=1.0, dtype="f32"):
        return (torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo).to(_TORCH[dtype])

    def byte(*shape):
        return torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)

    c = case
    if c["kind"] in ("add", "add_rows"):
        return {"a": uniform(c["rows"], c["cols"]), "b": uniform(c["rows"], c["cols"])}
    if c["kind"] == "softmax":
        return {"x": normal(c["rows"], c["cols"], std=2.0)}
    if c["kind"] == "layernorm":
        one = torch.ones((1, 1), device="cuda")
        return {"x": normal(c["rows"], c["cols"]), "gamma": uniform(1, c["cols"], lo=0.5, hi=1.5),
                "beta": normal(1, c["cols"], std=0.1), "inv_n": one / c["cols"], "eps": one * 1e-5}
    if c["kind"] == "matmul" and c["dtype"] == "i8":
        # results of about 40 a standard deviation: few of them saturate
        scale = 40.0 / (73.3 * 73.3 * math.sqrt(c["k"]))
        return {"a": byte(c["m"], c["k"]), "b": byte(c["k"], c["n"]),
                "scale": uniform(1, c["n"], lo=0.5 * scale, hi=1.5 * scale), "bias": uniform(1, c["n"], lo=-8, hi=8)}
    if c["kind"] == "matmul" and c["dtype"] == "f16":
        return {"a": uniform(c["m"], c["k"], dtype="f16"), "b": uniform(c["k"], c["n"], dtype="f16")}
    if c["kind"] == "matmul":
        return {"a": normal(c["m"], c["k"], std=0.02, dtype="bf16"), "b": normal(c["k"], c["n"], std=0.02, dtype="bf16")}
    if c["kind"] == "conv":
        src, filt = (c["n"], c["h"], c["w"], c["cin"]), (c["kh"], c["kw"], c["cin"], c["cout"])
        if c["dtype"] == "i8":
            return {"x": byte(*src), "f": byte(*filt)}
        return {"x": normal(*src, std=0.1, dtype=c["dtype"]), "f": normal(*filt, std=0.1, dtype=c["dtype"])}
    # queries carry the 1 / sqrt(d) of the scores
    return {"q": normal(c["heads"], c["nq"], c["d"], std=c["d"] ** -0.5, dtype=c["dtype"]),
            "k": normal(c["heads"], c["nk"], c["d"], dtype=c["dtype"]), "v": normal(c["heads"], c["nk"], c["d"])}


def _output(case):
    c = case
    if c["kind"] == "matmul":
        return (c["m"], c["n"]), "i8" if c["dtype"] == "i8" else "f32"
    if c["kind"] == "conv":
        return (c["n"], *_out_hw(c), c["cout"]), "f32"
    if c["kind"] == "attention":
        return (c["heads"], c["nq"], c["d"]), "f32"
    return (c["rows"], c["cols"]), "f32"


def prepare(case, seed):
    module = xt.compile(_module(case))
    inputs = _inputs(case, seed)
    shape, dtype = _output(case)
    out = torch.empty(shape, dtype=_TORCH[dtype], device="cuda")
    buffers = list(inputs.values())
    # memref order: results follow the operands, but an epilogue's and a
    # normalisation's parameters stand where their programs declare them
    at = 2 if case["kind"] == "matmul" else len(buffers)
    buffers.insert(at, out)
    return {"module": module, "buffers": buffers, "out": out}


def run(state):
    xt.launch(state["module"], *state["buffers"])
    return state["out"]


def work(case):
    c = case
    if c["kind"] == "matmul":
        size = _SIZE[c["dtype"]]
        moved = (c["m"] * c["k"] + c["k"] * c["n"]) * size
        moved += c["m"] * c["n"] + 8 * c["n"] if c["dtype"] == "i8" else 4 * c["m"] * c["n"]
        return {"bytes": moved, "flops": 2 * c["m"] * c["n"] * c["k"]}
    if c["kind"] == "conv":
        oh, ow = _out_hw(c)
        taps = c["kh"] * c["kw"] * c["cin"]
        moved = (c["n"] * c["h"] * c["w"] * c["cin"] + taps * c["cout"]) * _SIZE[c["dtype"]]
        pixels = c["n"] * oh * ow
        return {"bytes": moved + 4 * pixels * c["cout"], "flops": 2 * pixels * c["cout"] * taps}
    if c["kind"] == "attention":
        rows, keys, d = c["heads"] * c["nq"], c["heads"] * c["nk"], c["d"]
        return {"bytes": rows * d * (2 + 4) + keys * d * (2 + 4), "flops": 4 * rows * c["nk"] * d}
    n = c["rows"] * c["cols"]
    if c["kind"] in ("add", "add_rows"):
        return {"bytes": 12 * n, "flops": n}
    if c["kind"] == "softmax":
        return {"bytes": 8 * n, "flops": 5 * n}
    return {"bytes": 8 * n + 8 * c["cols"], "flops": 8 * n}


def tolerance(case):
    if case["kind"] in ("add", "add_rows") or _output(case)[1] == "i8":
        return "exact"  # one IEEE sum an element; whole numbers
    # about four times the error against 64 bits, which is 0.2 to 4 parts in
    # ten million where products are summed, less elsewhere
    summed = case["kind"] in ("matmul", "conv", "attention")
    return {"rel": 2e-6, "max": 5e-5} if summed else {"rel": 1e-6, "max": 2e-5}


def exact(case, seed):
    i = _inputs(case, seed)
    c = case
    if c["kind"] in ("add", "add_rows"):
        return i["a"].double() + i["b"].double()
    if c["kind"] == "softmax":
        return torch.softmax(i["x"].double(), dim=1)
    if c["kind"] == "layernorm":
        x = i["x"].double()
        x = x - x.sum(1, keepdim=True) * i["inv_n"].double()
        var = (x * x).sum(1, keepdim=True) * i["inv_n"].double()
        return x / torch.sqrt(var + i["eps"].double()) * i["gamma"].double() + i["beta"].double()
    if c["kind"] == "matmul":
        if c["dtype"] == "i8":
            return None  # whole numbers
        return i["a"].double() @ i["b"].double()
    if c["kind"] == "conv":
        oh, ow = _out_hw(c)
        ph, pw, s = c["kh"] // 2, c["kw"] // 2, c["stride"]
        x = torch.nn.functional.pad(i["x"].double(), (0, 0, pw, pw, ph, ph))
        out = torch.zeros((c["n"], oh, ow, c["cout"]), dtype=torch.float64, device="cuda")
        for a in range(c["kh"]):
            for b in range(c["kw"]):
                tap = x[:, a : a + (oh - 1) * s + 1 : s, b : b + (ow - 1) * s + 1 : s]
                out += (tap.reshape(-1, c["cin"]) @ i["f"][a, b].double()).view(out.shape)
        return out
    scores = i["q"].double() @ i["k"].double().transpose(1, 2).contiguous()
    return torch.softmax(scores, dim=2) @ i["v"].double()
