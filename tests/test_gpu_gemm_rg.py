"""GPU parity: MatMul of any size and alignment (gemm_rg) in each of its three block
forms, around the edges of its tiles, k steps and vector accesses."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from tests.gpu_util import dev, empty_dev, host, oracle_threads, say

pytestmark = pytest.mark.gpu

# batch, n, k, m
CASES = [
    # 64 x 64 tiles on two k groups: few rows, or few tiles in a batch; one k step (the
    # second group has none), two, an odd number, a last step of 1 and of 63
    (2, 33, 8, 4), (3, 64, 64, 5), (5, 65, 65, 67), (2, 1, 127, 130), (7, 100, 200, 63), (3, 17, 320, 61),
    (1, 40, 449, 9000), (1, 64, 16, 5001),
    # 128 x 64 tiles, an even and an odd number of steps, rows and columns around a tile
    (300, 65, 24, 12), (260, 70, 65, 9), (1, 1025, 33, 1000), (1, 2047, 191, 513), (1, 4097, 17, 130),
    (2, 1200, 100, 900),
    # 128 x 128 tiles with A in LDS: at least 512 of them and four steps
    (1, 2900, 200, 2950), (9, 1023, 257, 1021), (40, 400, 193, 500), (130, 250, 321, 251),
]


@pytest.mark.parametrize("batch,n,k,m", CASES)
def test_shapes(batch, n, k, m):
    """Full-range values (sums wrap), epilogues, gaps between batches' outputs, a
    broadcast B, operands at odd addresses; nothing outside the output is written."""
    g = wl.rng(940, batch, n, k, m)
    add, act = int(g.integers(0, 3)), int(g.integers(0, 3))
    gap, bcast, off = int(g.integers(0, 4)), bool(g.integers(0, 2)), int(g.integers(0, 5))
    say(f"gemm_rg {batch} x {n} x {k} x {m} add={add} act={act} gap={gap} bcast={bcast} offset={off}")
    full = lambda c: g.integers(-32768, 32768, c, dtype=np.int16)
    cs, bs = n * m + gap, 0 if bcast else k * m
    size = (batch - 1) * cs + n * m
    a, b = full(batch * n * k), full((1 if bcast else batch) * k * m)
    want = np.full(size, 0x5A5A, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.matmul(a, b, want, n, k, m, batch, n * k, bs, cs, threads=True)
    addv = full(m) if add == 2 else full(size) if add == 1 else None
    exp = want.astype(np.int32)
    for i in range(batch):
        v = exp[i * cs:i * cs + n * m]
        if add == 1:
            v += addv[i * cs:i * cs + n * m]
        elif add == 2:
            v += np.tile(addv, n)
        np.clip(v, -32768, 32767, out=v)
        if act:
            np.clip(v, 0, 32767 if act == 1 else 1536, out=v)

    def at_offset(v):
        t = empty_dev(off + v.size)
        t[off:] = dev(v)
        return t[off:]

    c = empty_dev(off + size + 64)
    K.MatmulKernel(at_offset(a), at_offset(b), c[off:off + size], n, k, m, batch, n * k, bs, cs,
                   add=None if addv is None else at_offset(addv), add_column=add == 2, act=act)
    got = host(c)
    np.testing.assert_array_equal(got[off:off + size].astype(np.int32), exp)
    assert (got[:off] == 0x5A5A).all() and (got[off + size:] == 0x5A5A).all()


@pytest.mark.parametrize("n,k,m", [(500, 1031, 600), (129, 2000, 2049), (300, 3001, 1000)])
def test_split(n, k, m):
    """A product of few tiles split over k through the workspace (odd k: ragged last
    step in the last split), against the unsplit call."""
    say(f"gemm_rg split {n} x {k} x {m}")
    g = wl.rng(941, n, k, m)
    a, b = g.integers(-32768, 32768, n * k, dtype=np.int16), g.integers(-32768, 32768, k * m, dtype=np.int16)
    want = np.zeros(n * m, np.int16)
    oracle.set_threads(oracle_threads())
    oracle.matmul(a, b, want, n, k, m, threads=True)
    need = K.matmul_workspace_size(n, k, m)
    assert need > 0
    for ws in (torch.full((need,), 0x5B, dtype=torch.uint8, device="cuda"), None):
        c = empty_dev(n * m)
        K.MatmulKernel(dev(a), dev(b), c, n, k, m, workspace=ws)
        np.testing.assert_array_equal(host(c), want)
