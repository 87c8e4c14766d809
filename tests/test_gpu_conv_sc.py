"""GPU parity: convolutions of at most four input channels (conv_sc): window widths
around a chunk of four columns, ragged rows and groups, int8 and wide weights, raw
and packed, up to several channel blocks and column blocks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from tests.gpu_util import dev, empty_dev, host, oracle_threads, say

pytestmark = pytest.mark.gpu

# N, C, H, W, M, kh, kw, stride, pt, pl, right padding
CASES = [
    (1, 3, 30, 40, 33, 7, 7, 2, 3, 3, 3), (2, 1, 9, 8, 40, 3, 3, 1, 1, 1, 1), (1, 4, 12, 9, 65, 2, 4, 1, 0, 0, 0),
    (2, 2, 17, 23, 34, 3, 5, 2, 2, 5, 0), (1, 3, 16, 33, 130, 1, 8, 1, 0, 4, 4), (1, 3, 21, 31, 48, 9, 3, 2, 4, 0, 1),
    (1, 3, 11, 600, 36, 3, 3, 2, 1, 1, 1), (2, 3, 8, 301, 50, 5, 5, 1, 2, 2, 2), (1, 4, 20, 16, 17, 8, 8, 1, 7, 7, 7),
    (3, 3, 40, 64, 96, 5, 1, 2, 2, 0, 0), (1, 1, 5, 13, 64, 4, 16, 1, 1, 8, 8),
]


@pytest.mark.parametrize("weights", ["int8", "mixed", "full"])
@pytest.mark.parametrize("N,C,H,W,M,kh,kw,s,pt,pl,pr", CASES)
def test_few_channels(N, C, H, W, M, kh, kw, s, pt, pl, pr, weights):
    g = wl.rng(860, N, C, H, W, M, kh, kw, s)
    OH, OW = (H + 2 * pt - kh) // s + 1, (W + pl + pr - kw) // s + 1
    act, off, bias = int(g.integers(0, 3)), int(g.integers(0, 5)), int(g.integers(0, 2))
    say(f"few channels {N}x{C}x{H}x{W} -> {M} {kh}x{kw} s{s} pt{pt} pl{pl} {weights} act={act} off={off} bias={bias}")
    full = lambda n: g.integers(-32768, 32768, n, dtype=np.int16)
    x, b = full(N * C * H * W), full(M)
    w = full(M * C * kh * kw) if weights == "full" else g.integers(-128, 128, M * C * kh * kw, dtype=np.int16)
    if weights == "mixed":     # one weight past int8 in one channel tile
        w[int(g.integers(0, w.size))] = int(g.choice([-129, 128, 32767, -32768]))
    args = (N, C, H, W, M, OH, OW, kh, kw, s, s, 1, 1, pt, pl, bias, 0)
    want = np.zeros(N * M * OH * OW, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    add = full(want.size) if g.integers(0, 2) else None
    exp = want.astype(np.int32) if add is None else np.clip(want.astype(np.int32) + add, -32768, 32767)
    if act:
        exp = np.clip(exp, 0, 32767 if act == 1 else 1536)

    def at_offset(v):
        t = empty_dev(off + v.size)
        t[off:] = dev(v)
        return t[off:]

    n = want.size
    addd = None if add is None else at_offset(add)
    y = empty_dev(off + n + 64)
    K.ConvKernel(at_offset(x), at_offset(w), dev(b), y[off:off + n], *args, add=addd, act=act)
    got = host(y)
    np.testing.assert_array_equal(got[off:off + n].astype(np.int32), exp)
    assert (got[:off] == 0x5A5A).all() and (got[off + n:] == 0x5A5A).all()
    size = K.conv_packed_size(*args)
    if size:
        packed = torch.empty(size, dtype=torch.uint8, device="cuda")
        K.conv_pack(dev(w), packed, *args)
        y2 = empty_dev(n)
        K.ConvPackedKernel(at_offset(x), packed, dev(b), y2, *args, add=addd, act=act)
        np.testing.assert_array_equal(host(y2).astype(np.int32), exp)
