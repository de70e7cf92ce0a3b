"""Products whose k loop runs in parts and whose m n outputs are any number: the partial products and the result then start
on the alignment of their elements only, and the last four outputs of a product may be fewer.  Against float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu

_T = {"bf16": t.bfloat16, "f32": t.float32}


def _component(nn):
    from i_amd import Component as i

    left = "bik*bkj~bijk" if nn else "bik*bjk~bijk"
    return i(f"{left} | i:16,j:16 | bjii'j'k") >> i("+bijk~bij | i:16,j:16 | bjii'j'k0")


# m n = 1, 2, 3 modulo 4, fewer than four outputs in all, one batch and several (whose results start anywhere)
@pytest.mark.parametrize("dtype, out", [("bf16", "f32"), ("bf16", "bf16"), ("f32", "f32")])
@pytest.mark.parametrize("nn", [False, True])
@pytest.mark.parametrize("b, m, n, k", [(1, 161, 211, 4022), (1, 3, 1, 3000), (3, 33, 41, 2048), (2, 17, 30, 4104), (1, 129, 127, 5000), (5, 1, 1, 1024),
                                        (1, 257, 259, 8192)])
def test_any_number_of_outputs(dtype, out, nn, b, m, n, k):
    component = _component(nn)
    g = t.Generator(device="cuda").manual_seed(m + n)
    x = t.randn(b, m, k, device="cuda", generator=g).to(_T[dtype])
    y = t.randn(*((b, k, n) if nn else (b, n, k)), device="cuda", generator=g).to(_T[dtype])
    xd, yd = x.double(), (y.double() if nn else y.double().transpose(1, 2).contiguous())
    ref = xd @ yd
    # f32 sums of k exact (bf16) or rounded (f32) products: a rounding per term, parts and lanes added on top; one of the result
    bound = (k + 64) * 2.0 ** -24 * (xd.abs() @ yd.abs()) + (2.0 ** -8 * ref.abs() if out == "bf16" else 0.0)
    for parts in (0, 2, 3, 7):
        component.option("gemm.k_parts", parts)
        for offset in (0, 1):
            ring = t.full((b * m * n + 32,), float("nan"), device="cuda", dtype=_T[out])
            c = ring[16 + offset:16 + offset + b * m * n].view(b, m, n)
            component.into(c, x, y)
            what = dict(dtype=dtype, out=out, nn=nn, b=b, m=m, n=n, k=k, parts=parts, offset=offset, report=component.report())
            assert bool(((c.double() - ref).abs() <= bound).all()), what
            assert bool(t.isnan(ring[:16 + offset]).all()) and bool(t.isnan(ring[16 + offset + b * m * n:]).all()), what
            assert parts == 0 or "parts)" in component.report(), what
