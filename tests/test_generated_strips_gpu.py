"""Generated nests in strips of four iterations and their bf16 forms: expressions without a kernel of their own, on
operands of f32 and bf16, lengths around multiples of four, views off a 16-byte boundary, outputs of either type and an
output that is its own input; against the same expression in float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


def _components():
    from i_amd import Component as i, I

    return {
        "column_normalize": ((I & i("+ij~j||ij")) >> i("ij/j~ij||1ij"), lambda x: x / x.sum(0, keepdim=True)),
        "column_max": (i(">ij~j"), lambda x: x.max(0).values),
        "column_sum": (i("+ij~j"), lambda x: x.sum(0)),
        "row_sum": (i("+ij~i"), lambda x: x.sum(1)),
        # (one nest, with a fused temporary that is private to every work-item)
        "staged_exponentials": (i("^ij~ij||ji") >> i("+ij~j||ji0"), lambda x: x.exp().sum(0)),
    }


_BITS = {t.float32: 0.0, t.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("types", ["f32-f32", "bf16-f32", "bf16-bf16", "f32-bf16"])
@pytest.mark.parametrize("name", ["column_normalize", "column_max", "column_sum", "row_sum", "staged_exponentials"])
def test_reductions_and_their_quotients(name, types):
    src, dst = ({"bf16": t.bfloat16, "f32": t.float32}[x] for x in types.split("-"))
    component, oracle = _components()[name]
    g = t.Generator(device="cuda").manual_seed(5)
    # columns: strips of a length below, at and around four; one work-item and many; rows: one, a few, several parts
    for rows, cols in [(1, 1), (3, 3), (5, 4), (7, 5), (64, 6), (33, 7), (200, 8), (1000, 63), (1001, 64), (999, 65), (4097, 130), (513, 1027), (2000, 2048), (300, 5001)]:
        for off in (0, 1, 2):
            buf = (0.1 + t.rand(rows * cols + 4, device="cuda", generator=g)).to(src)
            x = buf[off:off + rows * cols].view(rows, cols)
            ref = oracle(x.double())
            out_buf = t.full((ref.numel() + 8,), float("nan"), device="cuda", dtype=dst)
            out = out_buf[off:off + ref.numel()].view(ref.shape)
            component.into(out, x)
            # a sum of n positive terms in f32 is off by at most n 2^-24 of itself (in whatever order), a quotient by as
            # much and its own rounding, an exponential by two units in the last place; a bf16 result by one more rounding
            bound = ref.abs() * ((max(rows, cols) + 4) * 2.0 ** -24 + _BITS[dst])
            what = dict(name=name, types=types, rows=rows, cols=cols, off=off, report=component.report())
            assert bool(((out.double() - ref).abs() <= bound).all()), what
            assert bool(t.isnan(out_buf[:off]).all()) and bool(t.isnan(out_buf[off + ref.numel():]).all()), what


@pytest.mark.parametrize("src", ["f32", "bf16"])
def test_sums_of_few_rows_whose_strips_overlap(src):
    """Columns that are no multiple of four, too few rows for parts: neighbouring work-items, in other workgroups too,
    store the same sums of the columns they share.  Whole numbers: every sum is exact."""
    from i_amd import Component as i

    dtype = {"f32": t.float32, "bf16": t.bfloat16}[src]
    for expression, shapes in {"+ij~j": [(20, 257), (31, 515), (3, 5), (1, 1023), (20, 300001), (2, 1048579)],
                               "+bij~bj": [(5, 3, 255), (7, 20, 1021), (300, 4, 1001)]}.items():
        for shape in shapes:
            x = t.randint(-8, 9, shape, device="cuda").to(dtype)
            component = i(expression)
            ref = x.double().sum(-2).float()
            out = t.full_like(ref, float("nan"))
            for _ in range(3):
                component.into(out, x)
                assert t.equal(out, ref), dict(src=src, shape=shape, report=component.report())


@pytest.mark.parametrize("types", ["f32-f32", "bf16-f32", "bf16-bf16"])
def test_elementwise_with_a_broadcast_operand_and_a_scalar(types):
    from i_amd import Component as i

    src, dst = ({"bf16": t.bfloat16, "f32": t.float32}[x] for x in types.split("-"))
    component = i("ij+j~ij||ij") >> i("ij>.~ij||ij0")
    g = t.Generator(device="cuda").manual_seed(6)
    for rows, cols in [(1, 3), (2, 4), (9, 5), (100, 91), (77, 128), (500, 1023), (1200, 1024)]:
        x = t.randn(rows, cols, device="cuda", generator=g).to(src)
        b = t.randn(cols, device="cuda", generator=g).to(src)
        x[0, 0] = float("inf")
        x[0, cols - 1] = -float("inf")
        zero = t.zeros((), device="cuda")
        out = t.full((rows, cols), float("nan"), device="cuda", dtype=dst)
        component.into(out, x, b, zero)
        # one f32 sum, rounded once more where the result is bf16
        assert t.equal(out, t.clamp_min(x.float() + b.float(), 0.0).to(dst)), dict(types=types, rows=rows, cols=cols, report=component.report())


@pytest.mark.parametrize("dtype", [t.float32, t.bfloat16])
def test_an_output_that_is_its_own_input(dtype):
    """Strips of an odd length overlap, so an operand that is also the output takes the plain form there."""
    component, oracle = _components()["column_normalize"]
    for rows, cols in [(40, 64), (40, 65), (40, 67), (300, 1021)]:
        x = (0.1 + t.rand(rows, cols, device="cuda")).to(dtype)
        ref = oracle(x.double())
        component.into(x, x)
        assert bool(((x.double() - ref).abs() <= ref.abs() * ((rows + 4) * 2.0 ** -24 + _BITS[dtype])).all()), (rows, cols, component.report())


def test_rounding_to_bf16_is_to_nearest_even_and_keeps_nan():
    from i_amd import Component as i

    component = i("i+i~i")
    bits = t.arange(0, 1 << 16, device="cuda", dtype=t.int32)
    # every bf16 value, and the values just below, at and above the middle to the next one
    x = t.cat([(bits << 16) | low for low in (0, 0x7fff, 0x8000, 0x8001)]).view(t.float32)
    out = t.empty_like(x, dtype=t.bfloat16)
    component.into(out, x, t.zeros_like(x))
    want = (x + 0.0).to(t.bfloat16)
    assert t.equal(t.isnan(out), t.isnan(x))
    assert t.equal(out[~t.isnan(x)], want[~t.isnan(x)])


@pytest.mark.parametrize("static", [False, True])
def test_the_first_call_with_bf16_operands_may_be_under_capture(static):
    """A program that has run on f32 operands is captured on bf16 ones: the forms that read those are built then."""
    from i_amd import Component as i

    scaled, sums = i("ij+j~ij||ij") >> i("ij*.~ij||ij0"), i("+ij~j")
    two = t.full((), 2.0, device="cuda")
    x, b = t.randint(-8, 9, (300, 512), device="cuda").float(), t.randint(-8, 9, (512,), device="cuda").float()
    scaled.exec_torch(x, b, two)
    sums.exec_torch(x)
    xb, bb = x.bfloat16(), b.bfloat16()
    out, total = t.empty(300, 512, device="cuda", dtype=t.bfloat16), t.empty(512, device="cuda")
    t.cuda.synchronize()
    graph = t.cuda.CUDAGraph()
    with t.cuda.graph(graph):
        scaled.into(out, xb, bb, two, static_workspace=static)
        sums.into(total, xb, static_workspace=static)
    for _ in range(3):
        xb.copy_(t.randint(-8, 9, (300, 512), device="cuda"))
        out.zero_()
        total.zero_()
        t.cuda.synchronize()
        graph.replay()
        t.cuda.synchronize()
        assert t.equal(out, ((xb.float() + bb.float()) * 2).bfloat16()), scaled.report()
        assert t.equal(total, xb.float().sum(0)), sums.report()
