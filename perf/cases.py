"""The calls that are timed: what users of the framework have it do, each through the public entry points.

A case is a dict of plain values whose "path" names what is called:

  attention   mm_t >> scale >> row_max_shift >> exp >> row_normalize >> mm on [b, h, n, d] operands, in HBM
              (Component.into) or in host memory ("host": Component.exec_numpy, the reference's own way in)
  product     mm_t ("transposed": c = a b^T) or mm (c = a b), operands in HBM
  softmax     row softmax of [rows, cols]
  generated   expressions that have no kernel of their own and run as generated code

listed() holds one call of each kind of use, draw() gives others of the same ranges.
"""
import functools
import math

import numpy as np
import torch

from i_amd import Component as i, I

_TYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f32": 4}


# ---------------------------------------------------------------- the components
def _attention():
    s = "i:16,j:16"
    mm_t = i(f"bhik*bhjk~bhijk | {s} | bhjii'j'k") >> i(f"+bhijk~bhij | {s} | bhjii'j'k0")
    scale = i(f"bhij*.~bhij | {s} | bhji0i'j'")
    row_max_shift = (I & i(f">bhij~bhi | {s} | bhji0i'j'")) >> i(f"bhij-bhi~bhij | {s} | bhji01i'j'")
    exp = i(f"^bhij~bhij | {s} | bhji0i'j'")
    row_normalize = (I & i(f"+bhij~bhi | {s} | bhji0i'j'")) >> i(f"bhij/bhi~bhij | {s} | bhji01i'j'")
    mm = i(f"bhij*bhjk~bhikj | {s} | bhji0i'kj'") >> i(f"+bhikj~bhik | {s} | bhjii'kj'0")
    return mm_t >> scale >> row_max_shift >> exp >> row_normalize >> mm


def _product(transposed):
    if transposed:
        return i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    return i("ik*kj~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")


def _softmax():
    return (((I & i(">ij~i|i:16|ii'j")) >> i("ij-i~ij|i:16|ii'1j")) >> i("^ij~ij|i:16|ii'0j")
            >> ((I & i("+ij~i|i:16|ii'0j")) >> i("ij/i~ij|i:16|ii'01j")))


_GENERATED = {
    "column_normalize": lambda: (I & i("+ij~j||ij")) >> i("ij/j~ij||1ij"),
    "bias_relu": lambda: i("ij+j~ij||ij") >> i("ij>.~ij||ij0"),
    "column_sum": lambda: i("+ij~j"),
    "row_sum": lambda: i("+ij~i"),
}


@functools.lru_cache(maxsize=None)
def _component(path, which, f32_scale=False):
    """A program builds its components once and calls them with one operand after the other."""
    if path == "attention":
        component = _attention()
        return component.option("attention.f32_scale", 1) if f32_scale else component
    if path == "product":
        return _product(which)
    return _softmax() if path == "softmax" else _GENERATED[which]()


# ---------------------------------------------------------------- the cases
def _attention_case(dtype, b, h, nq, nk, d, out="f32", f32_scale=False, host=False):
    return {"path": "attention", "dtype": dtype, "b": b, "h": h, "nq": nq, "nk": nk, "d": d, "out": out, "f32_scale": f32_scale, "host": host}


def _product_case(dtype, transposed, m, n, k, out="f32"):
    return {"path": "product", "dtype": dtype, "transposed": transposed, "m": m, "n": n, "k": k, "out": out}


def _rows_case(path, dtype, rows, cols, out, which=""):
    return {"path": path, "which": which, "dtype": dtype, "rows": rows, "cols": cols, "out": out}


def listed():
    return [
        # the reference's demo at its small size: one f32 head, where launches and the way into the library count
        dict(_attention_case("f32", 1, 1, 512, 512, 64), name="demo"),
        # a whole batch of sequences in bf16: the benchmark's headline
        dict(_attention_case("bf16", 8, 32, 4096, 4096, 128), name="prefill"),
        # one new token of each sequence against the keys so far
        dict(_attention_case("bf16", 8, 32, 1, 4096, 128), name="decode"),
        # lengths and a head size that no tile divides, bf16 results for the next layer
        dict(_attention_case("bf16", 2, 12, 1000, 1000, 80, out="bf16"), name="ragged_attention"),
        # the reference's own interface: f32 arrays in host memory, one call that copies, runs and waits
        dict(_attention_case("f32", 8, 2, 2048, 2048, 64, host=True), name="host_attention"),
        # the large product
        dict(_product_case("bf16", True, 4096, 4096, 4096), name="mm_t"),
        # a product whose extents no tile or vector divides
        dict(_product_case("bf16", False, 2047, 3001, 777), name="ragged_mm"),
        # a layer applied to a few rows: the weights are read once
        dict(_product_case("bf16", True, 16, 8192, 8192, out="bf16"), name="narrow_mm_t"),
        # the reference's own type and layout
        dict(_product_case("f32", False, 1000, 1500, 700), name="mm_f32"),
        # the benchmark's row softmax
        dict(_rows_case("softmax", "f32", 16384, 4096, "f32"), name="softmax"),
        # rows of an odd length in bf16
        dict(_rows_case("softmax", "bf16", 4096, 5001, "bf16"), name="ragged_softmax"),
        # an expression of the user's own: columns divided by their sums
        dict(_rows_case("generated", "f32", 16384, 4096, "f32", "column_normalize"), name="column_normalize"),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _head_size(rng):
    return rng.choice([64, 128, 64, 128, 8 * rng.randint(4, 32)])


def _drawn(rng):
    use = rng.choice(["single", "prefill", "decode", "host", "product", "narrow", "softmax", "generated"])
    dtype = rng.choice(["bf16", "f32"])
    out = rng.choice(["bf16", "f32"]) if dtype == "bf16" else "f32"
    if use == "single":
        n = _spread(rng, 32, 2048)
        return _attention_case(dtype, 1, 1, n, n, 8 * rng.randint(4, 16), out)
    if use == "prefill":
        n = _spread(rng, 128, 16384)
        return _attention_case(dtype, _spread(rng, 1, 16), _spread(rng, 1, 32), n, n, min(_head_size(rng), 128 if dtype == "f32" else 256), out,
                               dtype == "bf16" and rng.random() < 0.25)
    if use == "decode":
        return _attention_case("bf16", _spread(rng, 1, 64), rng.randint(8, 64), _spread(rng, 1, 16), _spread(rng, 512, 32768), _head_size(rng),
                               rng.choice(["bf16", "f32"]))
    if use == "host":
        n = _spread(rng, 64, 2048)
        return _attention_case("f32", _spread(rng, 1, 8), rng.randint(1, 8), n, n, 8 * rng.randint(4, 16), host=True)
    if use == "product":
        return _product_case(dtype, rng.random() < 0.5, _spread(rng, 100, 8192), _spread(rng, 100, 8192), _spread(rng, 64, 8192), out)
    if use == "narrow":
        m, n, k = _spread(rng, 1, 64), 8 * _spread(rng, 128, 2048), 8 * _spread(rng, 128, 2048)
        return _product_case(dtype, rng.random() < 0.5, m, n, k, out)
    if use == "softmax":
        cols = _spread(rng, 16, 65536)
        return _rows_case("softmax", dtype, _spread(rng, 64, max(128, 2 ** 26 // cols)), cols, out)
    return _rows_case("generated", dtype, _spread(rng, 256, 16384), _spread(rng, 64, 4096), out, rng.choice(sorted(_GENERATED)))


def _affordable(case):
    """No more than the largest listed case: matrix work at the rate of its type, memory, and the host's link."""
    w = work(case)
    seconds = w["flops"] / (1.2e15 if case["dtype"] == "bf16" else 1.2e14) + w["bytes"] / (4e10 if case.get("host") else 4e12)
    return seconds < 1.5e-3


def draw(rng):
    case = _drawn(rng)
    while not _affordable(case):
        case = _drawn(rng)
    return case


# ---------------------------------------------------------------- one call
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, out = _TYPES[case["dtype"]], _TYPES[case["out"]]

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(dtype)

    def uniform(*shape):
        return torch.rand(*shape, device="cuda", generator=gen).to(dtype)

    path = case["path"]
    state = {"host": bool(case.get("host")), "component": _component(path, case.get("transposed", case.get("which")), case.get("f32_scale", False))}
    if path == "attention":
        b, h, nq, nk, d = (case[x] for x in ("b", "h", "nq", "nk", "d"))
        scale = torch.tensor(1.0 / math.sqrt(d), dtype=torch.float32, device="cuda")
        state["inputs"] = [normal(b, h, nq, d), normal(b, h, nk, d), scale, normal(b, h, nk, d)]
        shape = (b, h, nq, d)
    elif path == "product":
        m, n, k = case["m"], case["n"], case["k"]
        state["inputs"] = [normal(m, k), normal(n, k) if case["transposed"] else normal(k, n)]
        shape = (m, n)
    else:
        rows, cols = case["rows"], case["cols"]
        shape = {"column_sum": (cols,), "row_sum": (rows,)}.get(case["which"], (rows, cols))
        if case["which"] == "bias_relu":
            state["inputs"] = [normal(rows, cols), normal(cols), torch.zeros((), device="cuda")]
        else:  # sums of weights that are not negative, scores of either sign
            state["inputs"] = [uniform(rows, cols) if path == "generated" else normal(rows, cols)]
    if state["host"]:
        state["inputs"] = [x.cpu().numpy() for x in state["inputs"]]
    else:
        state["out"] = torch.empty(shape, dtype=out, device="cuda")
    return state


def run(state):
    if state["host"]:
        return state["component"].exec_numpy(*state["inputs"])
    return state["component"].into(state["out"], *state["inputs"])


# ---------------------------------------------------------------- what a call cannot do without, and how close results are
def work(case):
    e, o = _BYTES[case["dtype"]], _BYTES[case["out"]]
    if case["path"] == "attention":
        heads, nq, nk, d = case["b"] * case["h"], case["nq"], case["nk"], case["d"]
        return {"bytes": heads * d * (nq * (e + o) + 2 * nk * e), "flops": 4 * heads * nq * nk * d}
    if case["path"] == "product":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m + n) * k * e + m * n * o, "flops": 2 * m * n * k}
    rows, cols = case["rows"], case["cols"]
    written = {"column_sum": cols, "row_sum": rows}.get(case["which"], rows * cols)
    return {"bytes": rows * cols * e + written * o, "flops": 0}


def tolerance(case):
    """About four times the largest error seen against the same call in 64 bits, over the listed and sixty drawn cases."""
    if case["path"] == "attention" and case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.08}  # probabilities (and scaled queries) rounded to bf16: 2.9e-3 and 1.9e-2
    if case["out"] == "bf16":
        return {"rel": 1e-3, "max": 8e-3}  # f32 results that fall on either side of a rounding boundary: one unit of 2^-7
    if case["path"] in ("attention", "product"):
        return {"rel": 4e-6, "max": 4e-5}  # f32 sums in another order: 8.7e-7 and 8.5e-6
    return {"rel": 1e-6, "max": 5e-6}  # 1.2e-7 and 7.5e-7
