"""Products with few rows of A (at most 64): the kernels that stream B through registers.  Operands are small whole
numbers, so every sum is exact in f32 (below 2^24) in whatever order it is taken, and a bf16 result is that sum rounded
once: results are compared for equality with the product in float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


def _component(nn, b=""):
    from i_amd import Component as i

    right = f"{b}kj" if nn else f"{b}jk"
    return i(f"{b}ik*{right}~{b}ijk | i:16,j:16 | {b}jii'j'k") >> i(f"+{b}ijk~{b}ij | i:16,j:16 | {b}jii'j'k0")


@pytest.mark.parametrize("dtype, out", [("bf16", "bf16"), ("bf16", "f32"), ("f32", "f32")])
@pytest.mark.parametrize("nn", [False, True])
def test_products_of_few_rows(nn, dtype, out):
    types = {"bf16": t.bfloat16, "f32": t.float32}
    component = _component(nn)
    g = t.Generator(device="cuda").manual_seed(3)
    q = 8 if dtype == "bf16" else 4
    # k: one piece per wave and less, partial last pieces, several rounds of pieces; n: partial workgroups of 16, 32
    # and 64 columns, n that a 16-byte store cannot take (NT), grids of either workgroup size
    for m in (1, 7, 16, 17, 33, 64):
        for n in (512, 516, 1000, 16400) + (() if nn else (513, 1023)):
            for k in (512, 512 + q, 1000, 2048 + 3 * q, 4104):
                a = t.randint(-4, 5, (m, k), device="cuda", generator=g).to(types[dtype])
                b = t.randint(-4, 5, (k, n) if nn else (n, k), device="cuda", generator=g).to(types[dtype])
                buf = t.full((m * n + 8,), float("nan"), device="cuda", dtype=types[out])
                c = buf[:m * n].view(m, n)
                component.into(c, a, b)
                # (f32: NT up to 32 rows, NN always; bf16: NT up to 16 rows and 40 MB of B)
                narrow = (nn or m <= 32) if dtype == "f32" else not nn and m <= 16 and n * k <= 20_000_000
                assert ("_narrow" in component.report()) == narrow, (component.report(), m, n, k)
                ref = a.double() @ (b.double() if nn else b.double().t())
                assert t.equal(c, ref.to(types[out])), dict(nn=nn, dtype=dtype, out=out, m=m, n=n, k=k)
                assert bool(t.isnan(buf[m * n:]).all())


def test_values_of_b_that_no_row_of_the_tail_may_touch():
    """The partial last piece multiplies nothing: infinities just outside a row's end do not reach the sums."""
    component = _component(False)
    k, n = 520, 600
    wide = t.full((n, k + 64), float("inf"), device="cuda", dtype=t.bfloat16)
    b = wide.view(-1)[:n * k].view(n, k)
    b.fill_(1)
    a = t.ones(3, k, device="cuda", dtype=t.bfloat16)
    c = t.empty(3, n, device="cuda")
    component.into(c, a, b)
    assert t.equal(c, t.full_like(c, float(k)))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("nn", [False, True])
def test_batches_of_few_rows(nn, dtype):
    """Every batch reads its own operands, k whole and in parts (f32, row-major right operand); batches of whole slabs with
    many columns stay on the tiled kernels in bf16."""
    types = {"bf16": t.bfloat16, "f32": t.float32}
    component = _component(nn, "b")
    q = 8 if dtype == "bf16" else 4
    for b, m, n, k in [(2, 16, 512, 512), (3, 5, 516, 512 + q), (5, 12, 1000, 1000), (2, 31, 640, 2048 + 3 * q), (16, 16, 2048, 1024), (9, 1, 600, 4104)]:
        x = t.randint(-4, 5, (b, m, k), device="cuda").to(types[dtype])
        y = t.randint(-4, 5, (b, k, n) if nn else (b, n, k), device="cuda").to(types[dtype])
        c = t.full((b, m, n), float("nan"), device="cuda")
        component.into(c, x, y)
        ref = t.stack([x[s].double() @ (y[s].double() if nn else y[s].double().t()) for s in range(b)]).float()
        what = dict(nn=nn, dtype=dtype, b=b, m=m, n=n, k=k, report=component.report())
        assert t.equal(c, ref), what
        narrow = m <= 32 if dtype == "f32" else not nn and m <= 16 and not (b == 16 and n == 2048)
        assert ("_narrow" in component.report()) == narrow, what
