"""GPU parity: depthwise 3x3 / 5x5 streamed through registers, at the edges of its
row mapping (lanes per row, ragged rows, strips, tensors at odd addresses)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from tests.gpu_util import dev, empty_dev, host, oracle_threads, say

pytestmark = pytest.mark.gpu

# (window, stride, left padding) of every instance, and one that takes the band kernel
FORMS = [(3, 1, 0), (3, 1, 1), (3, 2, 0), (3, 2, 1), (5, 1, 2), (5, 2, 1), (5, 2, 2), (3, 1, 2)]
# one lane per row, a whole and a ragged last vector, one lane short of a wave,
# the widest row, and one column more (band kernel)
WIDTHS = [7, 8, 9, 15, 16, 33, 112, 117, 504, 505, 512, 513]


@pytest.mark.parametrize("k,s,pl", FORMS)
@pytest.mark.parametrize("W", WIDTHS)
def test_depthwise_rows(k, s, pl, W):
    """Full-range values (sums wrap), right padding of its own, out_ch < in_ch, an
    output and an Add operand at odd addresses; nothing past the output is written."""
    g = wl.rng(845, k, s, pl, W)
    N, C, M, H, pt, pr = 2, 4, 3, int(g.integers(k, 15)), int(g.integers(0, k)), int(g.integers(0, k))
    OH, OW = (H + 2 * pt - k) // s + 1, (W + pl + pr - k) // s + 1
    act, off = int(g.integers(0, 3)), int(g.integers(0, 9))
    say(f"depthwise rows {k}x{k} s{s} pl{pl} W={W} H={H} pt={pt} pr={pr} act={act} offset={off}")
    full = lambda n: g.integers(-32768, 32768, n, dtype=np.int16)
    x, w, b = full(N * C * H * W), full(M * k * k), full(M)
    args = (N, C, H, W, M, OH, OW, k, k, s, s, 1, 1, pt, pl, 1, 1)
    want = np.zeros(N * M * OH * OW, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    add = full(want.size)
    exp = np.clip(want.astype(np.int32) + add, -32768, 32767)
    if act != K.ACT_NONE:
        exp = np.clip(exp, 0, 32767 if act == K.ACT_RELU else 1536)
    n = want.size
    xd, addd, y = empty_dev(off + x.size), empty_dev(off + n), empty_dev(off + n + 64)
    xd[off:], addd[off:] = dev(x), dev(add)
    K.ConvKernel(xd[off:], dev(w), dev(b), y[off:off + n], *args, add=addd[off:], act=act)
    got = host(y)
    np.testing.assert_array_equal(got[off:off + n].astype(np.int32), exp)
    assert (got[:off] == 0x5A5A).all() and (got[off + n:] == 0x5A5A).all()


def test_depthwise_streaming_stores():
    """Tensors past the size from which the output is stored past the cache."""
    N, C, H = 8, 96, 216
    say("depthwise streaming stores")
    g = wl.rng(846)
    x, w, b = wl.uniform_q88(g, N * C * H * H, -4, 4), wl.normal_q88(g, C * 9, 0.4), wl.normal_q88(g, C, 0.1)
    args = (N, C, H, H, C, H, H, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    want = np.zeros(x.size, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    y = empty_dev(want.size)
    K.ConvKernel(dev(x), dev(w), dev(b), y, *args)
    np.testing.assert_array_equal(host(y), want)
