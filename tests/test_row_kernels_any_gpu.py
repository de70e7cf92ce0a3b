"""Rows of any length, alignment and type on the row kernels: softmax, row_max_shift, row_normalize and exp on
operands of f32 or bf16 on either side, against the same operation in float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu

_OPS = {
    "softmax": lambda t, x: t.softmax(x, dim=-1),
    "shift": lambda t, x: x - x.max(dim=-1, keepdim=True).values,
    "norm": lambda t, x: x / x.sum(dim=-1, keepdim=True),
    "exp": lambda t, x: t.exp(x),
}


def _component(op):
    from i_amd import Component as i, I

    if op == "softmax":
        return (((I & i(">ij~i|i:16|ii'j")) >> i("ij-i~ij|i:16|ii'1j")) >> i("^ij~ij|i:16|ii'0j")
                >> ((I & i("+ij~i|i:16|ii'0j")) >> i("ij/i~ij|i:16|ii'01j")))
    if op == "shift":
        return (I & i(">ij~i|i:16|ii'j")) >> i("ij-i~ij|i:16|ii'1j")
    if op == "norm":
        return (I & i("+ij~i|i:16|ii'j")) >> i("ij/i~ij|i:16|ii'1j")
    return i("^ij~ij")


# lengths around the edges of the groups (8 elements), of one lane, a wavefront, a workgroup and the longest row
# that registers hold (65536; 65537 takes two passes and, in bf16, f32 temporaries)
_COLS = [1, 2, 7, 8, 9, 15, 24, 31, 64, 65, 127, 129, 250, 255, 257, 498, 500, 513, 1023, 1530, 2049, 3001, 4082, 4083, 4090,
         4104, 5001, 6130, 8193, 12280, 16370, 16371, 24567, 30001, 49000, 65521, 65535, 65536, 65537]


@pytest.mark.parametrize("types", ["bf16-bf16", "bf16-f32", "f32-bf16", "f32-f32"])
@pytest.mark.parametrize("op", sorted(_OPS))
def test_rows_of_any_length_and_type(op, types):
    src, dst = ({"bf16": t.bfloat16, "f32": t.float32}[x] for x in types.split("-"))
    component = _component(op)
    g = t.Generator(device="cuda").manual_seed(11)
    for cols in _COLS:
        for rows, x_off, y_off in ((5, 0, 0), (9, 1, 1), (6, 3, 2)):
            n = rows * cols
            xbuf = (t.randn(n + 8, device="cuda", generator=g) if op != "norm" else t.rand(n + 8, device="cuda", generator=g)).to(src)
            ybuf = t.full((n + 16,), float("nan"), device="cuda", dtype=dst)
            x = xbuf[x_off:x_off + n].view(rows, cols)
            y = ybuf[y_off:y_off + n].view(rows, cols)
            component.into(y, x)
            ref = _OPS[op](t, x.double())
            # f32 arithmetic over a row (a sum of non-negative terms, an exponential and a product: a few 2^-23, the
            # exponent's own rounding up to 4 * 2^-23 included), and one rounding to nearest of a bf16 result
            bound = (ref.abs() + (1e-6 if op != "shift" else 1e-5)) * ((2.0 ** -8 if dst == t.bfloat16 else 0.0) + 4e-6)
            what = dict(op=op, types=types, rows=rows, cols=cols, x_off=x_off, y_off=y_off)
            assert bool(((y.double() - ref).abs() <= bound).all()), what
            assert bool(t.isnan(ybuf[:y_off]).all()) and bool(t.isnan(ybuf[y_off + n:]).all()), what


def test_rows_with_infinities_behave_as_the_float4_kernels():
    """A row of -inf only, one with +inf and one with a NaN give what the aligned f32 kernels give for them."""
    component = _component("softmax")
    x = t.randn(4, 64, device="cuda")
    x[0] = -float("inf")
    x[1, 3] = float("inf")
    x[2, 5] = float("nan")
    x[3, :60] = -float("inf")
    want = t.empty_like(x)
    component.into(want, x)
    for offset in (1, 2):
        xbuf = t.zeros(4 * 64 + 4, device="cuda")
        got = xbuf[offset:offset + 256].view(4, 64)
        got.copy_(x)
        out = t.empty(4 * 64 + 4, device="cuda")[offset:offset + 256].view(4, 64)
        component.into(out, got)
        assert t.allclose(out, want, rtol=1e-6, atol=0, equal_nan=True)
    out = t.empty(4, 64, device="cuda", dtype=t.bfloat16)
    component.into(out, x.bfloat16())
    same = t.empty_like(x)
    component.into(same, x.bfloat16().float())
    assert t.allclose(out.float(), same, rtol=2.0 ** -8, atol=0, equal_nan=True)
