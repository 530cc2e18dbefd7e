"""What the native training layer takes, as the library says on the host."""
import ctypes

import pytest

from na1d_amd import _lib, train


def _layer(dim=256, hidden=1024, heads=16, window=27, left=13, dilation=1, groups=1, ordered=0):
    return train._Layer(_lib.BF16, dim, hidden, heads, window, left, dilation, groups, ordered, 0.25)


@pytest.mark.parametrize("n,t,taken", [(1, 2, True), (65535, 2, True), (65536, 2, False), (1 << 19, 2, False), (65535, 16, True), (65536, 16, False),
                                       (1, 1 << 15, True), (1, 1 << 16, False), (1, 1, False), (0, 5, False)])
def test_sizes_that_launches_count(n, t, taken):
    c = _layer(heads=2)
    assert (_lib.load().na1d_train_layer_saved_bytes(ctypes.byref(c), n, t) > 0) == taken
