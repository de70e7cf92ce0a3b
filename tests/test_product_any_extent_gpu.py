"""Products of extents that no tile, vector or slab divides, in either layout and type: operands padded in one launch, row-major
right operands read as they are, outputs whose rows do not start on 16 bytes.  Operands are small whole numbers, so that
every sum is exact in f32 in whatever order it is taken: results are compared for equality with float64."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu

_TYPES = {"bf16": t.bfloat16, "f32": t.float32}


def _component(nn):
    from i_amd import Component as i

    if nn:
        return i("ik*kj~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    return i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")


def _check(nn, dtype, out, m, n, k, options=(), offset=0):
    g = t.Generator(device="cuda").manual_seed(m + 3 * n + 7 * k)
    component = _component(nn)
    for name, value in options:
        component = component.option(name, value)

    def whole(rows, cols):
        buf = t.full((rows * cols + 16,), float("inf"), device="cuda", dtype=_TYPES[dtype])  # (nothing outside takes part)
        x = buf[offset:offset + rows * cols].view(rows, cols)
        x.copy_(t.randint(-4, 5, (rows, cols), device="cuda", generator=g))
        return x

    a, b = whole(m, k), whole(k, n) if nn else whole(n, k)
    buf = t.full((m * n + 16,), float("nan"), device="cuda", dtype=_TYPES[out])
    c = buf[offset:offset + m * n].view(m, n)
    component.into(c, a, b)
    what = dict(nn=nn, dtype=dtype, out=out, m=m, n=n, k=k, options=options, offset=offset, report=component.report())
    assert t.equal(c, (a.double() @ (b.double() if nn else b.double().t())).to(_TYPES[out])), what
    assert bool(t.isnan(buf[:offset]).all()) and bool(t.isnan(buf[offset + m * n:]).all()), what
    return component.report()


@pytest.mark.parametrize("types", ["bf16-f32", "bf16-bf16", "f32-f32"])
@pytest.mark.parametrize("nn", [False, True])
def test_products_of_odd_extents(nn, types):
    dtype, out = types.split("-")
    for m, n, k in [(1, 1, 1), (3, 2, 5), (65, 63, 31), (64, 64, 64), (66, 130, 33), (127, 129, 100), (128, 132, 96), (130, 257, 777), (300, 301, 260),
                    (511, 515, 1001), (513, 1028, 520), (1000, 1500, 700)]:
        for offset in (0, 1):
            _check(nn, dtype, out, m, n, k, offset=offset)


@pytest.mark.parametrize("nn", [False, True])
def test_every_f32_tile_and_parts(nn):
    """The tiles that can be asked for, whole and partial slabs, k whole and in parts, at the edges of a tile and of a half
    of it.  (The 64 x 64 tile is the rule's own choice only: the tests below.)"""
    for tile in (0, 128, 256):
        for parts in (1, 3):
            for m, n, k in [(64, 64, 32), (63, 68, 36), (257, 260, 416), (129, 384, 1024), (128, 128, 256)]:
                report = _check(nn, "f32", "f32", m, n, k, options=(("gemm.tile", tile), ("gemm.k_parts", parts)))
                assert "gemm_nt_f32" in report and ("_brow" in report) == nn, report


def test_small_f32_tiles_are_reached():
    assert "64x64x32" in _check(True, "f32", "f32", 1000, 1500, 700)
    assert "64x64x32" in _check(False, "f32", "f32", 1000, 1500, 700)


@pytest.mark.parametrize("nn", [False, True])
def test_small_f32_tiles_in_parts(nn):
    """Few tiles under a long k: the rule takes 64-tiles in parts, whole and partial slabs in the last one."""
    for m, n, k in [(128, 128, 4096), (126, 132, 4092), (129, 68, 4100), (512, 64, 512), (500, 64, 516), (65, 100, 1288)]:
        report = _check(nn, "f32", "f32", m, n, k)
        assert "64x64x32" in report and "parts" in report and ("_brow" in report) == nn and ("_ktail" in report) == (k % 32 != 0), (m, n, k, report)


def test_an_f32_tile_that_is_asked_for_goes_in_parts_too():
    assert "256x256x32_direct (k in" in _check(False, "f32", "f32", 256, 256, 8192, options=(("gemm.tile", 256),))
    assert "128x128x32_direct (k in" in _check(False, "f32", "f32", 256, 256, 8192, options=(("gemm.tile", 128),))


def test_batched_row_major_right_operands_of_odd_extents():
    from i_amd import Component as i

    component = i("bik*bkj~bijk | i:16,j:16 | bjii'j'k") >> i("+bijk~bij | i:16,j:16 | bjii'j'k0")
    for dtype in (t.bfloat16, t.float32):
        for b, m, n, k in [(3, 70, 75, 33), (2, 130, 66, 264), (5, 64, 129, 77)]:
            x = t.randint(-4, 5, (b, m, k), device="cuda").to(dtype)
            y = t.randint(-4, 5, (b, k, n), device="cuda").to(dtype)
            c = t.full((b, m, n), float("nan"), device="cuda")
            component.into(c, x, y)
            ref = t.stack([x[s].double() @ y[s].double() for s in range(b)]).float()
            assert t.equal(c, ref), dict(dtype=dtype, b=b, m=m, n=n, k=k, report=component.report())


def test_only_the_operand_that_needs_padding_is_copied():
    """n alone is ragged: the right operand is copied, the left one, larger than the fixed workspace, is read as it is."""
    component = _component(True)
    for dtype, m, n, k in [(t.bfloat16, 8192, 1001, 8192), (t.float32, 8192, 333, 4096)]:
        a = t.randint(-4, 5, (m, k), device="cuda").to(dtype)
        b = t.randint(-4, 5, (k, n), device="cuda").to(dtype)
        c = t.full((m, n), float("nan"), device="cuda")
        component.into(c, a, b, static_workspace=True)
        rows = t.arange(0, m, 37, device="cuda")
        assert t.equal(c[rows], (a[rows].double() @ b.double()).float()), component.report()
        assert not bool(t.isnan(c).any())


def test_a_row_major_operand_of_more_elements_than_padding_can_copy_is_read_as_it_is():
    component = _component(True)
    m, n, k = 8, 16384, 1 << 19  # 2^33 elements
    a = t.randint(-4, 5, (m, k), device="cuda").bfloat16()
    b = t.ones(k, n, device="cuda", dtype=t.bfloat16)
    c = t.full((m, n), float("nan"), device="cuda")
    component.into(c, a, b, static_workspace=True)
    assert t.equal(c, a.double().sum(1).float()[:, None].expand(m, n)), component.report()
