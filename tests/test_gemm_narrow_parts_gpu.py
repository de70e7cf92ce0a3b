"""f32 products of few rows with a transposed right operand whose k loop is cut into parts over workgroups.  Operands are small
whole numbers, so every sum is exact in f32: results are compared for equality with float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


# few columns under a long k (as many parts as fill the chip), a ragged last part, columns and rows off the fragments, m n off
# four, more columns than one round of workgroups; and products that stay whole
@pytest.mark.parametrize("m, n, k, parts", [(3, 1688, 8896, True), (16, 1100, 6000, True), (17, 513, 5004, True), (31, 1024, 16000, True), (1, 515, 20000, True),
                                            (12, 4904, 6696, True), (32, 600, 1028, False), (30, 4096, 4096, False), (16, 8192, 2048, False)])
def test_parts_of_k(m, n, k, parts):
    from i_amd import Component as i

    component = i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    g = t.Generator(device="cuda").manual_seed(m + k)
    a = t.randint(-4, 5, (m, k), device="cuda", generator=g).float()
    wide = t.full((n * k + 64,), float("inf"), device="cuda")  # (nothing outside takes part)
    b = wide[:n * k].view(n, k)
    b.copy_(t.randint(-4, 5, (n, k), device="cuda", generator=g))
    ring = t.full((m * n + 8,), float("nan"), device="cuda")
    c = ring[:m * n].view(m, n)
    component.into(c, a, b)
    what = dict(m=m, n=n, k=k, report=component.report())
    assert t.equal(c, (a.double() @ b.double().t()).float()), what
    assert bool(t.isnan(ring[m * n:]).all()), what
    assert "_narrow" in component.report() and ("parts)" in component.report()) == parts, what


# 80, 81 and 85 column or output tiles: 240 workgroups in three parts are a round, 264 (the tiles of a part go up to a multiple of eight)
# are not, in the kernel for few rows and on 128-tiles
@pytest.mark.parametrize("m, n, k, three", [(2, 2560, 8000, True), (2, 2592, 8000, False), (1, 2713, 9001, False), (605, 2151, 3224, False), (601, 2050, 3001, False)])
def test_a_round_of_parts_holds_every_workgroup(m, n, k, three):
    from i_amd import Component as i

    component = i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    g = t.Generator(device="cuda").manual_seed(m + k)
    a, b = (t.randint(-4, 5, (rows, k), device="cuda", generator=g).float() for rows in (m, n))
    ring = t.full((m * n + 8,), float("nan"), device="cuda")
    c = ring[:m * n].view(m, n)
    component.into(c, a, b)
    what = dict(m=m, n=n, k=k, report=component.report())
    assert t.equal(c, (a.double() @ b.double().t()).float()), what
    assert bool(t.isnan(ring[m * n:]).all()), what
    crowded = "in 3 parts" in component.report() and "64x64" not in component.report()
    assert crowded == three, what
