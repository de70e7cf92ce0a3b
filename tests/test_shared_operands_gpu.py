"""Calls whose output shares memory with an input, in whole or in part, on the paths that read or store operands of 16 bits
where they lie: what such a call returned when they went through f32 copies is what it returns."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


def _i():
    from i_amd import Component as i, I

    return i, I


def _softmax():
    i, I = _i()
    s = "i:16,j:16"
    return (((I & i(f">ij~i|{s}|jii'j'")) >> i(f"ij-i~ij|{s}|1jii'j'")) >> i(f"^ij~ij|{s}|jii'j'")
            >> ((I & i(f"+ij~i|{s}|jii'j'")) >> i(f"ij/i~ij|{s}|1jii'j'")))


@pytest.mark.parametrize("j", [63, 64])
def test_an_output_in_another_order_than_its_input(j):
    i, _ = _i()
    x = t.randint(-99, 100, (40, 40, j), device="cuda").bfloat16()
    ref = (x.float() + x.float()).transpose(0, 1).to(t.bfloat16)
    component = i("bij+bij~ibj")
    component.into(x, x, x)
    assert t.equal(x, ref), component.report()


@pytest.mark.parametrize("j", [500, 511])
def test_an_input_that_is_read_again_after_an_output_in_its_place(j):
    i, _ = _i()
    for swapped in (False, True):
        x = t.randint(-9, 10, (300, j), device="cuda").bfloat16()
        doubled, sums = i("ij+ij~ij"), i("+ij~i")
        ref, total = (2 * x.float()).bfloat16(), x.double().sum(1).float()
        row = t.full((300,), float("nan"), device="cuda")
        component = (sums & doubled) if swapped else (doubled & sums)
        outputs, inputs = ([row, x], (x, x, x)) if swapped else ([x, row], (x, x, x))
        component.into(outputs, *inputs)
        assert t.equal(x, ref) and t.equal(row, total), (swapped, component.report())


@pytest.mark.parametrize("cols", [64, 1000, 5001])
def test_an_f32_output_over_a_bf16_input(cols):
    i, _ = _i()
    rows = 257
    buf = t.empty(rows, cols, device="cuda")
    x = buf.view(t.bfloat16).view(-1)[:rows * cols].view(rows, cols)
    x.copy_(t.randint(-9, 10, (rows, cols), device="cuda"))
    ref = 2 * x.float()
    component = i("ij+ij~ij")
    component.into(buf, x, x)
    assert t.equal(buf, ref), component.report()

    x.copy_(t.randn(rows, cols, device="cuda"))
    ref = t.softmax(x.double(), 1)
    component = _softmax()
    component.into(buf, x)
    # e^x through a 32-bit argument of at most 2^4, a sum of `cols` terms and a quotient
    assert bool(((buf - ref).abs() <= ref * ((cols + 32) * 2.0 ** -24)).all()), component.report()


@pytest.mark.parametrize("cols", [64, 1000, 5001])
@pytest.mark.parametrize("shift", [0, 1, 7])
def test_bf16_rows_over_themselves_and_over_other_rows(cols, shift):
    rows = 3000
    buf = t.randn(rows + shift, cols, device="cuda").bfloat16()
    x, out = buf[:rows], buf[shift:]
    ref = t.softmax(x.double(), 1)
    component = _softmax()
    component.into(out, x)
    assert bool(((out - ref).abs() <= ref * ((cols + 32) * 2.0 ** -24 + 2.0 ** -8)).all()), component.report()


@pytest.mark.parametrize("m, n, k", [(96, 100, 96), (600, 512, 600), (16, 1000, 512), (50, 4096, 1024)])
def test_an_f32_product_over_its_row_major_right_operand(m, n, k):
    i, _ = _i()
    component = i("ik*kj~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    a = t.randint(-4, 5, (m, k), device="cuda").float()
    b = t.randint(-4, 5, (k, n), device="cuda").float()
    ref = (a.double() @ b.double()).float()
    out = b.view(-1)[:m * n].view(m, n)
    component.into(out, a, b)
    assert t.equal(out, ref), component.report()


def test_an_f32_attention_of_large_heads_over_its_values():
    i, I = _i()
    s = "i:16,j:16"
    n, d = 700, 132
    mm_t = i(f"ik*jk~ijk | {s} | jii'j'k") >> i(f"+ijk~ij | {s} | jii'j'k0")
    row_max_shift = (I & i(f">ij~i | {s} | ji0i'j'")) >> i(f"ij-i~ij | {s} | ji01i'j'")
    exp = i(f"^ij~ij | {s} | ji0i'j'")
    row_normalize = (I & i(f"+ij~i | {s} | ji0i'j'")) >> i(f"ij/i~ij | {s} | ji01i'j'")
    mm = i(f"ij*jk~ikj | {s} | ji0i'kj'") >> i(f"+ikj~ik | {s} | jii'kj'0")
    component = mm_t >> row_max_shift >> exp >> row_normalize >> mm
    q, k, v = ((t.rand(n, d, device="cuda") - 0.5) for _ in range(3))
    ref = t.softmax(q.double() @ k.double().t(), 1) @ v.double()
    component.into(v, q, k, v)
    # scores up to 3 in f32 products of 132 terms, probabilities within as much, averages of values up to 1/2
    assert float((v - ref).abs().max()) <= (132 + 700 + 32) * 2.0 ** -24, component.report()
