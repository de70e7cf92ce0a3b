"""Calls on GPU tensors into caller-provided outputs: plain tensors are described in one array of words, everything else goes
the general way in, with the same results and the same refusals."""
import pytest
import torch as t

pytestmark = pytest.mark.gpu


def test_plain_tensors_and_everything_else_give_the_same():
    from i_amd import Component as i

    add = i("ij+j~ij||ij")
    x, b = t.randn(37, 19, device="cuda"), t.randn(19, device="cuda")
    want = x + b
    for xs, bs in ((x, b), (t.nn.Parameter(x), b), (x, t.nn.Parameter(b)), (x.clone().requires_grad_(), b)):
        out = t.full_like(want, float("nan"))
        assert add.into(out, xs, bs) is out
        assert t.equal(out, want)
    out = t.full_like(want, float("nan"))
    assert add.into([out], x, b) is out and t.equal(out, want)
    side = t.cuda.Stream()
    side.wait_stream(t.cuda.current_stream())
    with t.cuda.stream(side):
        add.into(out.zero_(), x, b)
    t.cuda.current_stream().wait_stream(side)
    assert t.equal(out, want)
    # rank 0, empty operands, two outputs
    scaled = i("i*.~i")
    y = t.empty(5, device="cuda")
    scaled.into(y, t.arange(5.0, device="cuda"), t.tensor(2.0, device="cuda"))
    assert t.equal(y, 2 * t.arange(5.0, device="cuda"))
    empty = t.empty(0, 19, device="cuda")
    assert add.into(empty, t.empty(0, 19, device="cuda"), b) is empty
    both = i("+ij~i") & i("+ij~j")
    r, c = t.empty(37, device="cuda"), t.empty(19, device="cuda")
    both.into((r, c), x)
    assert t.allclose(r, x.sum(1), atol=1e-5) and t.allclose(c, x.sum(0), atol=1e-5)


def test_refusals_stay():
    from i_amd import Component as i

    add = i("ij+j~ij||ij")
    x, b, out = t.randn(6, 4, device="cuda"), t.randn(4, device="cuda"), t.empty(6, 4, device="cuda")
    with pytest.raises(TypeError, match="contiguous"):
        add.into(out, t.randn(4, 6, device="cuda").t(), b)
    with pytest.raises(TypeError, match="contiguous"):
        add.into(t.empty(4, 6, device="cuda").t(), x, b)
    with pytest.raises(TypeError, match="float32 or bfloat16"):
        add.into(out, x.double(), b)
    with pytest.raises(TypeError, match="different places"):
        add.into(out, x.cpu(), b)
    with pytest.raises(RuntimeError, match="disagree on an index"):
        add.into(out, x, t.randn(5, device="cuda"))
    with pytest.raises(RuntimeError, match="inputs"):
        add.into(out, x)
    with pytest.raises(RuntimeError, match="wrong shape"):
        add.into(t.empty(6, 5, device="cuda"), x, b)
