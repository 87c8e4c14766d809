"""GPU parity: patch-GEMM convolutions whose input rows are not whole 16-byte groups
(the run staging): odd and even planes, groups over row and image ends, channels
that start between dwords, unread right columns, restaged chunks, single rows."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from tests.gpu_util import dev, empty_dev, host, oracle_threads, say

pytestmark = pytest.mark.gpu

# N, C, H, W, M, kh, kw, stride, dilation, pt, pl, right padding
CASES = [
    (3, 96, 7, 7, 96, 3, 3, 1, 1, 1, 1, 1), (2, 17, 9, 11, 70, 3, 3, 1, 1, 1, 1, 1),
    (2, 72, 14, 14, 80, 3, 3, 1, 1, 1, 1, 1), (3, 5, 13, 15, 66, 5, 5, 1, 1, 2, 2, 2),
    (2, 300, 14, 14, 40, 3, 3, 1, 1, 1, 1, 1), (1, 261, 7, 9, 129, 3, 3, 1, 1, 1, 1, 1),
    (2, 65, 20, 30, 70, 3, 2, 1, 1, 0, 0, 0), (1, 70, 31, 27, 68, 3, 3, 2, 1, 1, 1, 0),
    (1, 66, 12, 100, 65, 1, 3, 1, 1, 0, 2, 2), (4, 70, 5, 3, 66, 3, 3, 1, 1, 1, 1, 1),
    (2, 68, 1, 6, 72, 1, 2, 1, 1, 0, 1, 1), (2, 66, 23, 1, 66, 2, 1, 1, 1, 0, 0, 0),
    (1, 80, 18, 21, 70, 3, 3, 1, 2, 2, 2, 2), (2, 67, 6, 6, 65, 3, 3, 1, 1, 5, 4, 3),
    # several channel chunks on 32- and 64-row tiles, one patch and restaged
    (21, 70, 28, 28, 31, 3, 3, 1, 1, 1, 1, 1), (11, 130, 28, 27, 33, 3, 3, 1, 1, 1, 1, 1),
    (84, 600, 14, 14, 20, 3, 3, 1, 1, 1, 1, 1), (3, 81, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1),
    (1, 64, 15, 129, 96, 3, 3, 1, 1, 1, 1, 1), (2, 7, 63, 63, 90, 7, 7, 1, 1, 3, 3, 3),
]


@pytest.mark.parametrize("weights", ["int8", "full"])
@pytest.mark.parametrize("off", [0, 1, 2, 3])
@pytest.mark.parametrize("N,C,H,W,M,kh,kw,s,d,pt,pl,pr", CASES)
def test_run_staging(N, C, H, W, M, kh, kw, s, d, pt, pl, pr, off, weights):
    g = wl.rng(870, N, C, H, W, M, kh, kw, s, d, off)
    OH, OW = (H + 2 * pt - d * (kh - 1) - 1) // s + 1, (W + pl + pr - d * (kw - 1) - 1) // s + 1
    act, with_add = int(g.integers(0, 3)), int(g.integers(0, 2))
    say(f"runs {N}x{C}x{H}x{W} -> {M} {kh}x{kw} s{s} d{d} pt{pt} pl{pl} off={off} {weights} act={act} add={with_add}")
    full = lambda n: g.integers(-32768, 32768, n, dtype=np.int16)
    x, b = full(N * C * H * W), full(M)
    w = full(M * C * kh * kw) if weights == "full" else g.integers(-128, 128, M * C * kh * kw, dtype=np.int16)
    args = (N, C, H, W, M, OH, OW, kh, kw, s, s, d, d, pt, pl, 1, 0)
    want = np.zeros(N * M * OH * OW, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.conv(x, w, b, want, *args, threads=True)
    add = full(want.size) if with_add else None
    exp = want.astype(np.int32) if add is None else np.clip(want.astype(np.int32) + add, -32768, 32767)
    if act:
        exp = np.clip(exp, 0, 32767 if act == 1 else 1536)

    def at_offset(v):   # the tensor's bytes end with its last element
        t = empty_dev(off + v.size)
        t[off:] = dev(v)
        return t[off:]

    n = want.size
    y = empty_dev(off + n + 64)
    addd = None if add is None else at_offset(add)
    size = K.conv_packed_size(*args)
    if size:
        packed = torch.empty(size, dtype=torch.uint8, device="cuda")
        K.conv_pack(dev(w), packed, *args)
        K.ConvPackedKernel(at_offset(x), packed, dev(b), y[off:off + n], *args, add=addd, act=act)
    else:
        K.ConvKernel(at_offset(x), dev(w), dev(b), y[off:off + n], *args, add=addd, act=act)
    got = host(y)
    np.testing.assert_array_equal(got[off:off + n].astype(np.int32), exp)
    assert (got[:off] == 0x5A5A).all() and (got[off + n:] == 0x5A5A).all()
