"""TensorLayout.view against the index of every element's position (positions)."""
import numpy as np
import pytest

from cormorant_amd.scheduler.plan import TensorLayout


@pytest.mark.parametrize("lay", [
    TensorLayout.flat(1), TensorLayout.flat(37), TensorLayout.repeating(5, 8), TensorLayout.repeating(5, 24),
    TensorLayout.advancing(30, 3, 16), TensorLayout.advancing(30, 3, 10), TensorLayout.advancing(7, 7, 8),
    TensorLayout.advancing(12, 1, 16),
])
@pytest.mark.parametrize("extra", [0, 9])
def test_view_is_positions(lay, extra):
    buf = np.arange(1000, 1000 + lay.alloc + extra, dtype=np.int16)
    pos = lay.positions()
    np.testing.assert_array_equal(lay.view(buf).reshape(-1), buf[pos])
    data = np.arange(lay.numel, dtype=np.int16)
    want = buf.copy()
    want[pos] = data
    lay.view(buf)[...] = data.reshape(lay.view(buf).shape)
    np.testing.assert_array_equal(buf, want)


def test_view_stays_inside_the_buffer():
    with pytest.raises(ValueError):
        TensorLayout.advancing(30, 3, 16).view(np.zeros(41, np.int16))
