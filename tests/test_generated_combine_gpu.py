"""Generated sums in parts over work-items: the pass that puts the parts together, in one launch, into f32 or bf16, and the
strips of a nest that reads what another nest summed, at lengths that four does not divide.  Against float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu

_T = {"bf16": t.bfloat16, "f32": t.float32}


def _into(component, ref, terms, x, out, rows, parts=0):
    ring = t.full((ref.numel() + 32,), float("nan"), device="cuda", dtype=_T[out])
    y = ring[16:16 + ref.numel()].view(ref.shape)
    component.into(y, x)
    # a sum of `rows` f32 terms in any order, and one rounding to nearest of a bf16 result
    bound = rows * 2.0 ** -24 * terms + (2.0 ** -8 * ref.abs() if out == "bf16" else 0.0) + 1e-30
    what = dict(shape=tuple(x.shape), out=out, parts=parts, report=component.report())
    assert bool(((y.double() - ref).abs() <= bound).all()), what
    assert bool(t.isnan(ring[:16]).all()) and bool(t.isnan(ring[-16:]).all()), what


# buffers of one, a few, 63 to 65 and many elements (odd numbers leave a wavefront's last group of elements incomplete); parts on both
# sides of where the pass takes lanes at all (16) and more of them per element (65, 129, 257)
@pytest.mark.parametrize("dtype, out", [("f32", "f32"), ("bf16", "bf16"), ("bf16", "f32"), ("f32", "bf16")])
@pytest.mark.parametrize("cols", [1, 3, 63, 64, 65, 130, 1000])
def test_column_sums_in_any_number_of_parts(dtype, out, cols):
    from i_amd import Component as i

    component = i("+ij~j")
    g = t.Generator(device="cuda").manual_seed(cols)
    for rows in (64, 1100, 9000):
        x = t.randn(rows, cols, device="cuda", generator=g).to(_T[dtype])
        for parts in (0, 2, 15, 16, 17, 33, 64, 65, 128, 129, 256, 257, 511, 700):
            component.option("generated.parts", parts)
            _into(component, x.double().sum(0), x.double().abs().sum(0), x, out, rows, parts)
            assert parts == 0 or f" in {min(parts, rows)} parts" in component.report(), component.report()


@pytest.mark.parametrize("op, ref", [(">", lambda x: x.amax(0)), ("<", lambda x: x.amin(0)), ("*", lambda x: x.prod(0))])
def test_other_reductions(op, ref):
    from i_amd import Component as i

    component = i(f"{op}ij~j")
    x = 1.0 + t.rand(600, 77, device="cuda", generator=t.Generator(device="cuda").manual_seed(1)) * 0.01
    x[:, 5] = -x[:, 5]
    for parts in (2, 20, 300, 512):
        component.option("generated.parts", parts)
        want = ref(x.double())
        _into(component, want, want.abs(), x, "f32", 600, parts)
    x[17] = float("nan")
    if op == "*":
        assert bool(t.isnan(component.exec_torch(x)).all())


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_strips_of_a_nest_that_reads_another_nest_s_sums(dtype):
    from i_amd import Component as i, I

    component = (I & i("+ij~j||ij")) >> i("ij/j~ij||1ij")
    g = t.Generator(device="cuda").manual_seed(3)
    for rows, cols in ((100, 4), (300, 5), (257, 6), (64, 7), (1000, 333), (513, 1026)):
        x = (t.rand(rows, cols, device="cuda", generator=g) + 0.1).to(_T[dtype])
        ref = x.double() / x.double().sum(0)
        _into(component, ref, ref, x, dtype, rows + 2)  # (the quotient: the sum's error and two roundings)
        assert "strips of four" in component.report(), component.report()
    # the operand itself as the result: strips would overlap, so the nest runs as it is
    x = t.rand(129, 333, device="cuda", generator=g) + 0.1
    ref = x.double() / x.double().sum(0)
    component.into(x, x)
    assert bool(((x.double() - ref).abs() <= 131 * 2.0 ** -24 * ref).all())


def test_rows_of_64_and_more_are_a_wavefront_each():
    from i_amd import Component as i

    component = i("+ij~i")
    for cols, name in ((63, "f0_g"), (64, "f0_w"), (100, "f0_w")):
        x = t.rand(1000, cols, device="cuda")
        out = component.exec_torch(x)
        assert name in component.report(), component.report()
        assert bool(((out.double() - x.double().sum(1)).abs() <= cols * 2.0 ** -24 * x.double().sum(1)).all())
