"""The operators' autograd nodes in C++ (csrc/na1d_torch.cpp) against the Python Functions that serve what they leave."""
import pytest
import torch

from na1d_amd import _lib, dense, fused, nattn
from na1d_amd import na1d_fused, na1d_fused_qkv

pytestmark = pytest.mark.gpu


def _rand(*shape, dtype=torch.float16, seed=0, grad=True):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(dtype).cuda().requires_grad_(grad)


def _grads(out, leaves, g):
    return [out.detach(), *torch.autograd.grad(out, [t for t in leaves if t is not None and t.requires_grad], g)]


def _same(a, b):
    """The same kernels on the same operands: equal bits, except the bias gradient's float atomics (the order of a few
    hundred additions in fp32: 1e-4, and a unit of the result's type where that is 16 bit)."""
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype
        if x.dim() in (2, 4):
            torch.testing.assert_close(x, y, rtol=1e-4 if x.dtype == torch.float32 else 2.0 ** -10, atol=1e-4 * y.abs().max().item())
        else:
            assert torch.equal(x, y)


@pytest.mark.parametrize("bias", ["none", "fp32", "model", "fp16", "frozen"])
@pytest.mark.parametrize("dilation,p,lens", [(1, 0.0, None), (1, 0.2, "int32"), (3, 0.0, "int64"), (2, 0.1, None)])
@pytest.mark.parametrize("N,H,T,C,W,left", [(3, 2, 50, 24, 27, 13), (1, 1, 1, 8, 3, 1), (2, 4, 130, 32, 65, 32), (2, 3, 37, 128, 4, 0)])
def test_fused_nodes_are_the_python_functions(N, H, T, C, W, left, dilation, p, lens, bias):
    q, k, v = (_rand(N * H, T, C, seed=i) for i in range(3))
    shape = {"model": (1, H, 1, W)}.get(bias, (H, W))
    rpb = None if bias == "none" else _rand(*shape, dtype=torch.float16 if bias == "fp16" else torch.float32, seed=5, grad=bias != "frozen")
    t_valid = None if lens is None else torch.randint(1, T + 1, (N,), generator=torch.Generator().manual_seed(1)).to(getattr(torch, lens)).cuda()
    drop = (p, -5) if p else None                    # seeds wrap to 64 bits either way
    g = _rand(N * H, T, C, seed=9, grad=False)
    out = _lib.nodes().fused(q, k, v, rpb, t_valid, H, W, left, 0.3, dilation, *fused._native_dropout(drop))
    assert out is not None
    want = fused._FusedNA1D.apply(q, k, v, rpb, t_valid, H, W, left, 0.3, False, dilation, drop)
    _same(_grads(out, (q, k, v, rpb), g), _grads(want, (q, k, v, rpb), g))
    qkv, g = _rand(N, T, 3, H, C, seed=3), _rand(N, T, H * C, seed=9, grad=False)
    out = _lib.nodes().fused_qkv(qkv, rpb, t_valid, W, left, 0.3, dilation, *fused._native_dropout(drop))
    want = fused._FusedNA1DQKV.apply(qkv, rpb, t_valid, W, left, 0.3, False, dilation, drop)
    _same(_grads(out, (qkv, rpb), g), _grads(want, (qkv, rpb), g))
    with torch.no_grad():                             # without a node: no log-sum-exp either
        assert torch.equal(_lib.nodes().fused_qkv(qkv, rpb, t_valid, W, left, 0.3, dilation, *fused._native_dropout(drop)), want)


@pytest.mark.parametrize("B,H,T,C,p", [(4, 2, 70, 64, 0.0), (3, 1, 200, 40, 0.2), (2, 2, 1, 8, 0.0)])
def test_dense_and_two_call_nodes_are_the_python_functions(B, H, T, C, p):
    q, k, v, g = (_rand(B, T, C, dtype=torch.bfloat16, seed=i) for i in range(4))
    t_valid = torch.full((B // H,), max(1, T - 3), dtype=torch.int32).cuda()
    out = _lib.nodes().dense(q, k, v, t_valid, H, 0.2, p, 7)
    want = dense._GlobalAttention.apply(q, k, v, t_valid, H, 0.2, (p, 7) if p else None)
    _same(_grads(out, (q, k, v), g.detach()), _grads(want, (q, k, v), g.detach()))
    QK, AV = nattn.getNA1dFunction(C, 1, torch.bfloat16)
    python = torch.autograd.Function.apply.__func__
    attn = QK.apply(q, k, 5, 2, 1)
    assert "Python" not in type(attn.grad_fn).__name__ and not isinstance(attn.grad_fn, torch.autograd.function.BackwardCFunction)
    ga = torch.randn(B, T, 5, device="cuda")
    want = python(QK, q, k, 5, 2, 1)
    for x, y in zip(_grads(attn, (q, k), ga), _grads(want, (q, k), ga)):
        assert torch.equal(x, y)
    a = torch.softmax(attn.detach(), -1).requires_grad_(True)
    for x, y in zip(_grads(AV.apply(a, v, 5, 2, 1), (a, v), g.detach()), _grads(python(AV, a, v, 5, 2, 1), (a, v), g.detach())):
        assert torch.equal(x, y)


def test_nodes_leave_what_they_do_not_take_to_python():
    q, k, v = (_rand(2, 20, 16, seed=i) for i in range(3))
    nodes = _lib.nodes()

    def take(q=q, k=k, v=v, rpb=None, t_valid=None, H=1, W=5, left=2, dilation=1, p=0.0):
        return nodes.fused(q, k, v, rpb, t_valid, H, W, left, 1.0, dilation, p, 0)
    assert take() is not None
    wide = _rand(2, 20, 136)
    assert take(q=q.transpose(0, 1)) is None and take(k=k.float()) is None and take(v=v.cpu()) is None and take(k=k[:, :10]) is None
    assert take(H=3) is None and take(W=81, left=0) is None and take(left=5) is None and take(dilation=0) is None and take(p=1.0) is None
    assert take(q=wide, k=wide, v=wide) is None and take(rpb=_rand(1, 4, dtype=torch.float32)) is None
    assert take(t_valid=torch.ones(3, dtype=torch.int32).cuda()) is None
    with pytest.raises(AssertionError):
        na1d_fused(q.transpose(1, 2), k, v, 5, 2)
    assert na1d_fused(wide, wide, wide, 5, 2).shape == wide.shape                    # the generic kernels
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: na1d_fused(a, a, a, 5, 2))(torch.stack([q.detach(), k.detach()]))
    with torch.autograd.forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        dual = torch.autograd.forward_ad.make_dual(q.detach(), torch.ones_like(q))
        na1d_fused(dual, dual, dual, 5, 2)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = na1d_fused(q, k, v, 5, 2)
    assert len(seen) >= 5
    a, b = _grads(out, (q, k, v), torch.ones_like(q)), _grads(na1d_fused(q, k, v, 5, 2), (q, k, v), torch.ones_like(q))
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    out = na1d_fused(q, k, v, 5, 2)
    with torch.no_grad():
        q.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    qkv = _rand(2, 20, 3, 1, 16)
    old = _lib.load().na1d_force_generic(1)
    try:
        assert nodes.fused_qkv(qkv, None, None, 5, 2, 1.0, 1, 0.0, 0) is None and na1d_fused_qkv(qkv, 5, 2).shape == (2, 20, 16)
    finally:
        _lib.load().na1d_force_generic(old)


def _dirty(*shape):
    """Leaves numbers in the memory that the next allocation of this size gets."""
    for t in [torch.full(shape, 3.0, device="cuda") for _ in range(8)]:
        del t


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("N,H,T,C,W,left,dilation,p", [(2, 16, 100, 16, 27, 13, 1, 0.0), (1, 1, 1, 8, 3, 1, 1, 0.0), (3, 5, 150, 32, 65, 32, 1, 0.0),
                                                       (1, 12, 3, 64, 80, 40, 2, 0.1), (2, 7, 33, 24, 15, 7, 3, 0.0)])
def test_bias_gradient_begins_at_zero(N, H, T, C, W, left, dilation, p, in_place):
    """The forward's kernel clears the sums of a node's first backward; backwards of a kept graph, and captured ones, clear their own."""
    rpb = eager = _rand(1, H, 1, W, dtype=torch.float32, seed=5)
    tensors = [_rand(N, T, 3, H, C, seed=3)] if in_place else [_rand(N * H, T, C, seed=i) for i in range(3)]
    g = _rand(*((N, T, H * C) if in_place else (N * H, T, C)), seed=9, grad=False)

    def call():
        _dirty(1, H, 1, W)
        if in_place:
            return _lib.nodes().fused_qkv(tensors[0], rpb, None, W, left, 0.3, dilation, p, 11)
        return _lib.nodes().fused(*tensors, rpb, None, H, W, left, 0.3, dilation, p, 11)

    if in_place:
        out = fused._FusedNA1DQKV.apply(*tensors, rpb, None, W, left, 0.3, False, dilation, (p, 11) if p else None)
    else:
        out = fused._FusedNA1D.apply(*tensors, rpb, None, H, W, left, 0.3, False, dilation, (p, 11) if p else None)
    want = torch.autograd.grad(out, rpb, g)[0]
    out, other = call(), call()
    for n in range(3):                               # the first is kept unchanged while the second runs
        first, second = (torch.autograd.grad(o, rpb, g, retain_graph=n < 2)[0] for o in (out, other))
        for got in (first, second):
            torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4 * want.abs().max().item())     # float atomics, as in _same
    kept = call()
    # Leaves of the graph's own: the engine joins the stream on which a leaf was first used, which must be a captured one.
    rpb, tensors = rpb.detach().clone().requires_grad_(True), [t.detach() for t in tensors]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = torch.autograd.grad(call(), rpb, g)[0]
    for _ in range(3):
        graph.replay()
        torch.testing.assert_close(captured, want, rtol=1e-4, atol=1e-4 * want.abs().max().item())
    torch.testing.assert_close(torch.autograd.grad(kept, eager, g)[0], want, rtol=1e-4, atol=1e-4 * want.abs().max().item())


@pytest.mark.parametrize("in_place", [False, True])
def test_bias_gradient_under_compiled_autograd(in_place):
    """Which copies a node's data, also for a graph that is walked twice."""
    from torch._dynamo import compiled_autograd
    N, H, T, C, W = 2, 4, 50, 32, 15
    rpb = _rand(H, W, dtype=torch.float32, seed=5)
    tensors = [_rand(N, T, 3, H, C, seed=3)] if in_place else [_rand(N * H, T, C, seed=i) for i in range(3)]
    g = _rand(*((N, T, H * C) if in_place else (N * H, T, C)), seed=9, grad=False)

    def call():
        _dirty(H, W)
        return na1d_fused_qkv(*tensors, W, 7, rpb=rpb, scale=0.3) if in_place else na1d_fused(*tensors, W, 7, rpb=rpb, num_heads=H, scale=0.3)

    call().backward(g)
    want = rpb.grad
    with compiled_autograd._enable(lambda graph: torch.compile(graph, backend="eager")):
        out, other = call(), call()
        for o, keep in ((out, True), (other, False), (out, True), (out, False)):
            rpb.grad = None
            o.backward(g, retain_graph=keep)
            torch.testing.assert_close(rpb.grad, want, rtol=1e-4, atol=1e-4 * want.abs().max().item())     # float atomics, as in _same
