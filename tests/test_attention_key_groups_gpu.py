"""bf16 attention whose workgroups cut the keys into parts over groups of wavefronts, against float64."""
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


def _bound(q, k, v, scale, p):
    """What roundings to bf16 (half a unit of 2^-8 each) may do: to the scaled queries, hence to a score by 2^-9 of its absolute
    terms, on both sides of the division; to the probabilities, and to the result."""
    terms = (q.abs() @ k.abs().transpose(1, 2) * abs(scale)).amax(-1, keepdim=True)
    return (2.0 ** -8 * terms + 2.0 ** -7) * (p @ v.abs()) + 2.0 ** -8 * (p @ v).abs() + 1e-6


def _check(component, q, k, v, scale, kernel, out_dtype=t.float32):
    bh, nq, dv = q.shape[0], q.shape[1], v.shape[2]
    ring = t.full((bh * nq * dv + 64,), float("nan"), device="cuda", dtype=out_dtype)
    out = ring[32:32 + bh * nq * dv].view(bh, nq, dv)
    component.into(out, q, k, t.tensor(scale, device="cuda"), v)
    q, k, v = (x.double() for x in (q, k, v))
    p = t.softmax(q @ k.transpose(1, 2) * scale, -1)
    what = dict(q=tuple(q.shape), k=tuple(k.shape), v=tuple(v.shape), scale=scale, report=component.report())
    assert bool(((out.double() - p @ v).abs() <= _bound(q, k, v, scale, p)).all()), what
    assert bool(t.isnan(ring[:32]).all()) and bool(t.isnan(ring[-32:]).all()), what
    assert (kernel in component.report()) if kernel else ("_k" not in component.report().split()[1]), what


def _operands(bh, nq, nk, d, dv, seed):
    g = t.Generator(device="cuda").manual_seed(seed)
    return [t.randn(bh, n, w, device="cuda", generator=g).bfloat16() for n, w in ((nq, d), (nk, d), (nk, dv))]


# kernel, d, dv, key counts at the edges of its tiles and groups: fewer tiles in some groups, a partial last one, long enough
# for the steady loop in every group
@pytest.mark.parametrize("kernel, d, dv, keys", [
    ("d64_bn32_direct_w1_k8 ", 64, 64, (513, 768, 1000, 1279, 1600, 2047)),
    ("d64_bn32_direct_w1_k8_pad ", 40, 56, (544, 1025, 1601)),
    ("d128_bn32_direct_w2_k4 ", 128, 128, (513, 640, 1023, 1535, 2040)),
    ("d128_bn32_direct_w2_k4_pad ", 80, 96, (515, 608, 1300)),
    ("d128_bn32_direct_w2_k4_pad ", 72, 128, (515, 608, 1300)),
    ("d256_bn32_direct_w2_k2 ", 256, 256, (700, 1024, 1501)),
    ("d256_bn32_direct_w2_k2_pad ", 136, 184, (737, 1024, 1501)),
])
def test_edges_of_tiles_and_groups(kernel, d, dv, keys):
    component = _component()
    for nk in keys:
        for bh, nq, out in ((1, 1, t.float32), (3, 33, t.bfloat16), (2, 65, t.float32), (5, 64, t.bfloat16)):
            print("case", kernel, bh, nq, nk, flush=True)
            q, k, v = _operands(bh, nq, nk, d, dv, nk + nq)
            name = kernel.strip() if "_pad" not in kernel or max(d, dv) > 96 or max(d, dv) <= 64 else kernel.strip() + " (96 columns)"
            _check(component, q, k, v, d ** -0.5, name, out)
            _check(component, q, k, v, -0.4 * d ** -0.5, name, out)
    q, k, v = _operands(2, 40, keys[0], d, dv, 1)
    _check(component, q, k, v, 0.0, "_k")


def test_two_waves_and_four_groups_at_head_size_64():
    component = _component()
    for bh, nq, nk, d in ((8, 1536, 1537, 64), (12, 1000, 1281, 48), (100, 100, 2047, 64)):
        q, k, v = _operands(bh, nq, nk, d, d, nk)
        _check(component, q, k, v, d ** -0.5, "d64_bn64_direct_w2_k4")


@pytest.mark.parametrize("d", [64, 128])
def test_groups_whose_scores_lie_far_apart(d):
    """The keys of one group score far above or below the others: the pass without a reference is done again with the running
    max, and the groups' sums differ by up to 2^430; or they score -inf, and weigh nothing."""
    component = _component()
    nk = 1536
    for offset in (80.0, -300.0, -float("inf")):
        q, k, v = _operands(2, 70, nk, d, d, 3)
        q, k = q * 0.5, k * 0.5
        q[:, :, 0] = 1.0
        k[:, :, 0] = 0.0
        k[:, 384:768, 0] = offset
        if offset > -1e30:
            _check(component, q, k, v, 1.0, "_k")
            continue
        out = component.exec_torch(q, k, t.tensor(1.0, device="cuda"), v)
        keep = t.cat([t.arange(384), t.arange(768, nk)]).cuda()
        q, k, v = q.double(), k[:, keep].double(), v[:, keep].double()
        p = t.softmax(q @ k.transpose(1, 2), -1)
        worst = float(((out.double() - p @ v).abs() / _bound(q, k, v, 1.0, p)).max())
        assert worst <= 1.0, worst
    out = component.exec_torch(q.bfloat16(), t.full((2, nk, d), -float("inf"), device="cuda").bfloat16(), t.tensor(1.0, device="cuda"), t.ones(2, nk, d, device="cuda").bfloat16())
    assert bool(t.isnan(out).all())


# few and many groups, and one group of all keys (head size 64 asks for it with a tile)
@pytest.mark.parametrize("d, nq, kernel, options", [(64, 70, "_w1_k8", {}), (48, 70, "_w1_k8", {}), (64, 1500, "_w2_k4", {}), (128, 70, "_w2_k4", {}), (256, 70, "_w2_k2", {}),
                                                    (64, 70, "_direct", {"attention.kv_parts": 1}), (56, 300, "_direct", {"attention.kv_parts": 1})])
@pytest.mark.parametrize("offset", [-2e2, -2e3, -3e4, -1e9, t.finfo(t.bfloat16).min, -float("inf")])
def test_first_tiles_far_below_the_rest(d, nq, kernel, options, offset):
    """Masked keys are the first tile of a group, or the first of all, or both: the groups start on a reference far below
    the scores that follow."""
    component = _component()
    for name, value in options.items():
        component.option(name, value)
    nk = 1792
    q, k, v = _operands(8 if nq > 1000 else 2, nq, nk, d, d, 4)
    q, k = q * 0.5, k * 0.5
    q[:, :, 0] = 1.0
    k[:, :, 0] = 0.0
    # (tiles of 64 and 32 keys; groups of 224, 448 and 896)
    for masked in ([(0, 64)], [(896, 960)], [(224, 288), (448, 512), (1344, 1408)], [(0, 64), (896, 1200)]):
        k2, keep = k.clone(), t.ones(nk, dtype=t.bool, device="cuda")
        for first, last in masked:
            k2[:, first:last, 0] = offset
            keep[first:last] = False
        out = component.exec_torch(q, k2, t.tensor(1.0, device="cuda"), v)
        assert kernel in component.report() and (not options or "_k" not in component.report().split()[1]), component.report()
        q64, k64, v64 = q.double(), k[:, keep].double(), v[:, keep].double()  # (e^-200 weighs nothing)
        p = t.softmax(q64 @ k64.transpose(1, 2), -1)
        # (_bound, with the terms of the keys that weigh something)
        worst = float(((out.double() - p @ v64).abs() / _bound(q64, k64, v64, 1.0, p)).max())
        assert worst <= 1.0, (masked, worst, component.report())


def test_who_asks_for_another_kernel_gets_it():
    q, k, v = _operands(2, 100, 1200, 128, 128, 5)
    for name, value in (("attention.kv_parts", 1), ("attention.f32_scale", 1), ("attention.waves", 4)):
        component = _component()
        component.option(name, value)
        _check(component, q, k, v, 128 ** -0.5, "")
    big = _operands(300, 1, 1200, 128, 128, 6)  # more workgroups than CUs
    _check(_component(), *big, 128 ** -0.5, "")
