"""What the native training layer takes, as the library says on the host."""
import ctypes

import pytest
import torch

from na1d_amd import _lib, models, train


def _layer(dim=256, hidden=1024, heads=16, window=27, left=13, dilation=1, groups=1, ordered=0):
    return train._Layer(_lib.BF16, dim, hidden, heads, window, left, dilation, groups, ordered, 0.25)


@pytest.mark.parametrize("n,t,taken", [(1, 2, True), (65535, 2, True), (65536, 2, False), (1 << 19, 2, False), (65535, 16, True), (65536, 16, False),
                                       (1, 1 << 15, True), (1, 1 << 16, False), (1, 1, False), (0, 5, False)])
def test_sizes_that_launches_count(n, t, taken):
    c = _layer(heads=2)
    assert (_lib.load().na1d_train_layer_saved_bytes(ctypes.byref(c), n, t) > 0) == taken


@pytest.mark.parametrize("change,fits", [
    (lambda bn: None, True), (lambda bn: bn._buffers.update(num_batches_tracked=torch.zeros((), dtype=torch.int32)), False),
    (lambda bn: bn._buffers.update(num_batches_tracked=torch.zeros((), dtype=torch.float32)), False),
    (lambda bn: bn._buffers.update(num_batches_tracked=bn.num_batches_tracked.to("meta")), False),
    (lambda bn: bn._buffers.update(num_batches_tracked=None), False), (lambda bn: bn._buffers.update(running_mean=None), False),
    (lambda bn: bn._buffers.update(running_var=bn.running_var.to("meta")), False), (lambda bn: bn.double(), False),
    (lambda bn: bn._buffers.update(running_mean=torch.zeros(8)), False)])
def test_a_norm_whose_counters_the_kernels_cannot_write(change, fits):
    """The kernel adds one to eight bytes on the layer's device; torch's statistics take what they are given there."""
    bn = models.BatchNorm1d(256)
    change(bn)
    assert train._norm_fits(bn, 256, torch.device("cpu")) == fits


def _pooling(context, pooled, seed=0):
    """Pooling as a model has it, in 64 bits: the logits are made from x by way of the context."""
    gen = torch.Generator().manual_seed(seed)
    x, w = torch.randn(2, 8, 9, generator=gen, dtype=torch.float64).requires_grad_(True), torch.randn(8, 24, generator=gen, dtype=torch.float64)
    rows = x * 1.0
    return x, pooled(torch.tanh(w @ context(rows)), rows), torch.randn(2, 16, generator=gen, dtype=torch.float64)


_NODES = (lambda x: train._Context.apply(x, 1e-12), lambda z, x: train._Pooled.apply(z, x, 1e-12))
_OPERATIONS = (lambda x: train.context_of(x, 1e-12)[0], lambda z, x: train.pooled_of(z, x, 1e-12))


@pytest.mark.filterwarnings("ignore:.*autocast")
def test_pooling_gradients_that_are_differentiated_again():
    """Where one input of a node is made from the other, its gradient counts once; the same sums in 64 bits."""
    results = []
    for nodes in (_NODES, _OPERATIONS):
        x, out, d = _pooling(*nodes)
        (dx,) = torch.autograd.grad(out, x, d, create_graph=True)
        results.append((dx, torch.autograd.grad(dx.square().sum(), x, create_graph=True)[0]))
    for got, want in zip(*results):
        assert torch.allclose(got, want, rtol=1e-10, atol=1e-10 * float(want.abs().max()))


@pytest.mark.filterwarnings("ignore:.*autocast")
def test_pooling_gradients_in_batches():
    """Several gradients at once (is_grads_batched; jacobian with vectorize), as torch's operations take them; 64 bits."""
    results = []
    for nodes in (_NODES, _OPERATIONS):
        x, out, d = _pooling(*nodes)
        results.append(torch.autograd.grad(out, x, torch.stack([d, d.flip(0), 2 * d]), is_grads_batched=True)[0])
    assert torch.allclose(*results, rtol=1e-10, atol=1e-10)


@pytest.mark.filterwarnings("ignore:.*autocast")
def test_pooling_outputs_can_be_written_to():
    """What the nodes return is the caller's, as what torch's operations return is; 64 bits."""
    results = []
    for context, pooled in (_NODES, _OPERATIONS):
        x, out, d = _pooling(lambda rows: context(rows).mul_(0.5), lambda z, rows: pooled(z, rows).mul_(3).add_(1))
        results.append((out, torch.autograd.grad(out, x, d, create_graph=True)[0]))
    assert torch.equal(results[0][0], results[1][0]) and torch.allclose(results[0][1], results[1][1], rtol=1e-10, atol=1e-10)
