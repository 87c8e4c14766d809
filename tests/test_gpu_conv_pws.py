"""GPU parity: pointwise convolutions on eight-pixel groups (conv_pws), at the edges
of its tiles: channels around a k step and around its two block forms, planes that
are not whole groups, few and odd output channels, tensors at odd addresses."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from tests.gpu_util import dev, empty_dev, host, oracle_threads, say

pytestmark = pytest.mark.gpu

# in_ch, pixels, out_ch, images: pixels not a multiple of 8 (or more than 256
# channels) take the path from 2^19 (2^20) outputs on
CASES = [
    (8, 8, 1, 1), (8, 16, 17, 3), (9, 64, 16, 2), (63, 24, 33, 5), (64, 1000, 40, 2), (65, 136, 64, 3),
    (128, 8, 130, 40), (255, 72, 15, 9), (256, 520, 48, 1),
    (16, 9, 600, 100), (24, 49, 110, 100), (40, 3025, 36, 5), (130, 15, 400, 90),
    (257, 16, 1100, 61), (320, 49, 214, 101), (511, 24, 700, 63), (512, 201, 300, 18),
]


@pytest.mark.parametrize("bias", [0, 1])
@pytest.mark.parametrize("C,P,M,N", CASES)
def test_pointwise_groups(C, P, M, N, bias):
    """Full-range values (sums wrap) with every epilogue; nothing past the output is written."""
    g = wl.rng(850, C, P, M, N, bias)
    act, add, off = int(g.integers(0, 3)), bool(g.integers(0, 2)), int(g.integers(0, 9))
    say(f"pointwise groups C={C} P={P} M={M} N={N} bias={bias} act={act} add={add} offset={off}")
    full = lambda n: g.integers(-32768, 32768, n, dtype=np.int16)
    x, w, b = full(N * C * P), full(M * C), full(M)
    args = (N, C, P, 1, M, P, 1, 1, 1, 1, 1, 1, 1, 0, 0, bias, 0)
    n = N * M * P
    want = np.zeros(n, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    exp = want.astype(np.int32)
    a = full(n) if add else None
    if add:
        exp = np.clip(exp + a, -32768, 32767)
    if act != K.ACT_NONE:
        exp = np.clip(exp, 0, 32767 if act == K.ACT_RELU else 1536)

    def at_offset(v):
        t = empty_dev(off + v.size)
        t[off:] = dev(v)
        return t[off:]

    y = empty_dev(off + n + 64)
    K.ConvKernel(at_offset(x), at_offset(w), dev(b), y[off:off + n], *args, add=at_offset(a) if add else None, act=act)
    got = host(y)
    np.testing.assert_array_equal(got[off:off + n].astype(np.int32), exp)
    assert (got[:off] == 0x5A5A).all() and (got[off + n:] == 0x5A5A).all()


@pytest.mark.parametrize("P", [1024, 1023])
def test_pointwise_in_place_add(P):
    """The residual is the output tensor itself; tensors past the cached size."""
    N, C, M = 70, 64, 256
    say(f"pointwise in-place add P={P}")
    g = wl.rng(851, P)
    x, w, b = wl.uniform_q88(g, N * C * P, -2, 2), wl.normal_q88(g, M * C, 0.2), wl.normal_q88(g, M, 0.1)
    args = (N, C, P, 1, M, P, 1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 0)
    want = np.zeros(N * M * P, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    res = wl.uniform_q88(g, want.size, -3, 3)
    y = dev(res)
    K.ConvKernel(dev(x), dev(w), dev(b), y, *args, add=y, act=K.ACT_RELU)
    np.testing.assert_array_equal(host(y).astype(np.int32), np.clip(want.astype(np.int32) + res, 0, 32767))
