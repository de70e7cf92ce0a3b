"""f32 attention with 16 query rows per workgroup and the keys in parts over its wavefronts, against float64."""
import math

import pytest
import torch as t

pytestmark = pytest.mark.gpu


def _component():
    from i_amd import Component as i, I

    s = "i:16,j:16"
    return ((i(f"bik*bjk~bijk | {s} | bjii'j'k") >> i(f"+bijk~bij | {s} | bjii'j'k0")) >> i(f"bij*.~bij | {s} | bji0i'j'")
            >> ((I & i(f">bij~bi | {s} | bji0i'j'")) >> i(f"bij-bi~bij | {s} | bji01i'j'")) >> i(f"^bij~bij | {s} | bji0i'j'")
            >> ((I & i(f"+bij~bi | {s} | bji0i'j'")) >> i(f"bij/bi~bij | {s} | bji01i'j'"))
            >> (i(f"bij*bjk~bikj | {s} | bji0i'kj'") >> i(f"+bikj~bik | {s} | bjii'kj'0")))


def _reference(q, k, v, scale):
    """The result in float64 and what f32 arithmetic may be off by: a score by (d + 2) roundings of its absolute terms, a
    weight by that, the exponential's 4 and its argument's one, on both sides of the division, a sum by one rounding per key."""
    q, k, v = (x.double() for x in (q, k, v))
    s = q @ k.transpose(1, 2) * scale
    p = t.softmax(s, -1)
    terms = (q.abs() @ k.abs().transpose(1, 2) * abs(scale)).amax(-1, keepdim=True)
    eps = 2.0 ** -24
    weight = ((q.shape[-1] + 4) * terms + 8) * eps
    return p @ v, (2 * weight + k.shape[1] * eps) * (p @ v.abs()) + 1e-30


def _check(component, bh, nq, nk, d, dv, scale, seed=0, waves=True):
    g = t.Generator(device="cuda").manual_seed(seed)
    q, k, v = (t.randn(bh, n, w, device="cuda", generator=g) for n, w in ((nq, d), (nk, d), (nk, dv)))
    ring = t.full((bh * nq * dv + 32,), float("nan"), device="cuda")
    out = ring[16:16 + bh * nq * dv].view(bh, nq, dv)
    component.into(out, q, k, t.tensor(scale, device="cuda"), v)
    ref, bound = _reference(q, k, v, scale)
    what = dict(bh=bh, nq=nq, nk=nk, d=d, dv=dv, scale=scale, report=component.report())
    assert bool(((out.double() - ref).abs() <= bound).all()), what
    assert bool(t.isnan(ring[:16]).all()) and bool(t.isnan(ring[-16:]).all()), what
    assert ("_waves" in component.report()) == waves, what


@pytest.mark.parametrize("d, dv", [(64, 64), (128, 128), (4, 4), (20, 36), (48, 64), (68, 4), (96, 96), (124, 128)])
def test_edges_of_the_tile_the_steps_and_the_rows(d, dv):
    component = _component()
    for nq, nk in ((1, 129), (15, 256), (16, 257), (17, 511), (33, 1000), (300, 145), (5, 640)):
        for bh in (1, 3):
            print("case", d, dv, nq, nk, bh, flush=True)
            _check(component, bh, nq, nk, d, dv, 1.0 / math.sqrt(d), seed=nq + nk)
    _check(component, 2, 40, 300, d, dv, -0.3)
    _check(component, 2, 40, 300, d, dv, 0.0)


def test_keys_also_in_parts_over_workgroups():
    component = _component()
    for bh, nq, nk, d in ((1, 5, 4100, 64), (2, 40, 8192, 128), (1, 64, 5000, 100)):
        _check(component, bh, nq, nk, d, d, d ** -0.5)
        assert " x " in component.report().split("(keys in")[1], component.report()


def test_who_asks_for_a_tile_kernel_gets_it():
    component = _component()
    component.option("attention.kv_parts", 1)
    _check(component, 1, 300, 300, 64, 64, 0.125, waves=False)
    component.option("attention.kv_parts", 2)
    _check(component, 1, 300, 300, 64, 64, 0.125, waves=False)
    component.option("attention.kv_parts", 0)
    _check(component, 64, 2048, 96, 64, 64, 0.125, waves=False)  # a grid that fills the chip


def test_scores_of_minus_infinity_infinity_and_nan():
    """Keys that score -inf weigh nothing wherever they lie (a whole part of them too); a row of nothing else, +inf or a NaN
    gives NaN, as subtracting the maximum does."""
    component = _component()
    q = t.zeros(1, 4, 64, device="cuda")
    q[0, :, 0] = 1.0
    k = t.randn(1, 512, 64, device="cuda", generator=t.Generator(device="cuda").manual_seed(1))
    v = t.randn(1, 512, 64, device="cuda", generator=t.Generator(device="cuda").manual_seed(2))
    k[0, 64:200, 0] = -float("inf")
    out = component.exec_torch(q, k, t.tensor(1.0, device="cuda"), v)
    assert "_waves8" in component.report()
    keep = t.cat([t.arange(64), t.arange(200, 512)]).cuda()
    ref, bound = _reference(q, k[:, keep], v[:, keep], 1.0)
    assert bool(((out.double() - ref).abs() <= bound).all())
    for bad in (float("inf"), float("nan")):
        k2 = k.clone()
        k2[0, 300, 0] = bad
        assert bool(t.isnan(component.exec_torch(q, k2, t.tensor(1.0, device="cuda"), v)).all()), bad
    k[0, :, 0] = -float("inf")
    assert bool(t.isnan(component.exec_torch(q, k, t.tensor(1.0, device="cuda"), v)).all())


# (bh, nq, nk, d): every shape goes into several parts over workgroups
@pytest.mark.parametrize("bh, nq, nk, d", [(1, 16, 8192, 32), (1, 64, 4096, 20), (64, 1, 1024, 32), (1, 5, 4100, 64), (200, 1, 4096, 64), (1, 64, 5000, 128)])
def test_parts_over_workgroups_that_score_minus_infinity_weigh_nothing(bh, nq, nk, d):
    """Whole parts at the end, at the beginning and in the middle; where every part is so, the row is NaN."""
    component = _component()
    g = t.Generator(device="cuda").manual_seed(nk)
    q = t.randn(bh, nq, d, device="cuda", generator=g)
    q[:, :, 0] = 1.0
    k, v = (t.randn(bh, nk, d, device="cuda", generator=g) for _ in range(2))
    one = t.tensor(1.0, device="cuda")
    for first, last in ((nk // 3, nk), (0, nk - 40), (nk // 8, nk // 8 * 7)):
        k2 = k.clone()
        k2[:, first:last, 0] = -float("inf")
        out = component.exec_torch(q, k2, one, v)
        assert " x " in component.report().split("(keys in")[1], component.report()
        keep = t.cat([t.arange(first), t.arange(last, nk)]).cuda()
        ref, bound = _reference(q, k[:, keep], v[:, keep], 1.0)
        assert bool(((out.double() - ref).abs() <= bound).all()), (first, last, component.report())
    k[:, :, 0] = -float("inf")
    assert bool(t.isnan(component.exec_torch(q, k, one, v)).all())


@pytest.mark.parametrize("bh, nq, nk, d", [(48, 700, 700, 64), (1, 300, 700, 32), (1, 64, 512, 128), (1, 64, 4096, 32), (200, 1, 4096, 64)])
@pytest.mark.parametrize("scale", [1.0, 3.0, 0.125])
def test_scores_of_the_lowest_value_weigh_nothing(bh, nq, nk, d, scale):
    """Times log2(e) they are beyond f32 from a scale of 0.7 on.  They lie on the keys of whole wavefronts, and of whole parts over
    workgroups where there are such."""
    component = _component()
    g = t.Generator(device="cuda").manual_seed(d)
    q = t.randn(bh, nq, d, device="cuda", generator=g)
    q[:, :, 0] = 1.0
    k, v = (t.randn(bh, nk, d, device="cuda", generator=g) for _ in range(2))
    for first, last in ((nk // 2, nk), (0, nk // 2)):
        for low in (t.finfo(t.float32).min, t.finfo(t.bfloat16).min):
            k2 = k.clone()
            k2[:, first:last, 0] = low
            out = component.exec_torch(q, k2, t.tensor(scale, device="cuda"), v)
            assert "_waves" in component.report()
            keep = t.cat([t.arange(first), t.arange(last, nk)]).cuda()
            ref, bound = _reference(q, k[:, keep], v[:, keep], scale)
            assert bool(((out.double() - ref).abs() <= bound).all()), (first, low, component.report())
