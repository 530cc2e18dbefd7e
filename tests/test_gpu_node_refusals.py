"""Calls that the autograd nodes' kernels refuse: the Python functions run them, or refuse them as they always did."""
import pytest
import torch

from na1d_amd import _lib, na1d_fused, na1d_fused_qkv
from na1d_amd.dense import global_attention
from na1d_amd.nattn import getNA1dFunction

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.float16).cuda()


def _misaligned(*shape):
    n = torch.Size(shape).numel()
    return _rand(n + 8)[1:n + 1].view(shape)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("T,dilation", [(87400, 1), (81400, 64)])
def test_rows_too_far_apart_for_one_launch(T, dilation, grad):
    """Rows of 16 heads of 128 channels, read in place, end where 32-bit offsets do at some 87000 of them; longer
    sequences, and dilated ones from 81000 on, go through packed copies."""
    H, C, W, left = 16, 128, 9, 4
    qkv = torch.randn(1, T, 3, H, C, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda", dtype=torch.float16)
    rpb = _rand(H, W).float()
    packed = [qkv[:, :, i].permute(0, 2, 1, 3).contiguous().view(H, T, C).requires_grad_(grad) for i in range(3)]
    qkv.requires_grad_(grad)
    out = na1d_fused_qkv(qkv, W, left, rpb=rpb, scale=0.1, dilation=dilation)
    want = na1d_fused(*packed, W, left, rpb=rpb, num_heads=H, scale=0.1, dilation=dilation)
    assert torch.equal(out.view(T, H, C).transpose(0, 1), want)
    if grad:
        g = _rand(T, H, C)
        (dqkv,) = torch.autograd.grad(out, qkv, g.view(1, T, H * C))
        for i, d in enumerate(torch.autograd.grad(want, packed, g.transpose(0, 1).contiguous())):
            assert torch.equal(dqkv[0, :, i].transpose(0, 1), d)


def test_refusals_are_na1d_errors():
    q, k, v = (_rand(2, 20, 16, seed=i) for i in range(3))
    bad = _misaligned(2, 20, 16)
    QK, AV = getNA1dFunction(16, 1, torch.float16)
    attn = torch.rand(2, 20, 5, device="cuda")
    for grad in (False, True):
        qg = q.clone().requires_grad_(grad)
        for call in (lambda: na1d_fused(qg, bad, v, 5, 2), lambda: na1d_fused(qg, k, v, 5, 2, scale=0.0), lambda: na1d_fused(qg, k, v, 5, 2, scale=float("nan")),
                     lambda: na1d_fused(qg, k, bad, 5, 2, dilation=2), lambda: na1d_fused_qkv(_misaligned(2, 20, 3, 1, 16).requires_grad_(grad), 5, 2),
                     lambda: na1d_fused_qkv(_rand(2, 20, 3, 1, 16).requires_grad_(grad), 5, 2, scale=-1.0),
                     lambda: global_attention(qg, bad, v, 1), lambda: global_attention(qg, k, v, 1, scale=-1.0),
                     lambda: QK.apply(qg, bad, 5, 2, 1), lambda: AV.apply(attn, bad, 5, 2, 1)):
            with pytest.raises(_lib.NA1DError):
                call()


def test_refusals_in_the_backward_are_na1d_errors():
    q, k, v = (_rand(2, 20, 16, seed=i).requires_grad_(True) for i in range(3))
    QK, AV = getNA1dFunction(16, 1, torch.float16)
    attn = torch.rand(2, 20, 5, device="cuda", requires_grad=True)
    grads = _misaligned(2, 20, 16)
    for out in (na1d_fused(q, k, v, 5, 2), na1d_fused(q, k, v, 5, 2, dilation=2), global_attention(q, k, v, 1), AV.apply(attn, v, 5, 2, 1)):
        with pytest.raises(_lib.NA1DError, match="failed"):
            out.backward(grads)
        assert q.grad is None
    na1d_fused(q, k, v, 5, 2).backward(grads.clone())
    assert torch.isfinite(q.grad).all()
