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
