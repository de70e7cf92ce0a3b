"""Products with few rows of A (at most 64): the kernels that stream B through registers.  Operands are small whole
numbers, so every sum is exact in f32 (below 2^24) in whatever order it is taken, and a bf16 result is that sum rounded
once: results are compared for equality with the product in float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


def _component(nn):
    from i_amd import Component as i

    if nn:
        return i("ik*kj~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    return i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")


@pytest.mark.parametrize("out", ["bf16", "f32"])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("nn", [False, True])
def test_products_of_few_rows(nn, dtype, out):
    if dtype == "f32" and out == "bf16":
        pytest.skip("an f32 product of this program has an f32 result")
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
