"""GPU split/merge where its hull bounds and its block sizes have edges.

Boundaries must equal the oracle's exact-sum split/merge: whole numbers, no
tolerance.  Minimum sizes: 64 and 127 (one ballot, odd rows), 128 (the widest
block), 129 and 131 (no block size: sums only), 256, 300 and 1000 (2, 3 and 8
blocks per unit), 1016 (127 * 8, the widest window), 1100 (11 units of 100: sums
only).  Data: noise of 0 or 1 (a power of two next to the bound), convex runs (more
hull vertices than a block keeps), values at and around +-2^52 (the exact range's
ends, some blocks outside it), residuals at powers of two, unsigned values whose
fitted lines go below zero."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def data(kind, n, seed):
    r = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    if kind == "noise1":
        return (i * 3 + r.integers(0, 2, n)).astype(np.int32)
    if kind == "convex":
        return ((i % 3000 - 1500) ** 2 // 7 + 5).astype(np.uint32)
    if kind == "edge52":
        return ((1 << 52) - 2 * n + i * 3 + r.integers(0, 9, n)).astype(np.int64)
    if kind == "below52":
        return (-(1 << 52) + i * 5 - r.integers(0, 9, n) * (i % 2000 < 700)).astype(np.int64)
    if kind == "mixed":
        return (np.where((i // 700) % 4 == 1, 1 << 56, 0) + i * 11 + r.integers(0, 99, n)).astype(np.uint64)
    if kind == "pow2":
        return (i * 5 + r.integers(-64, 65, n) + 64).astype(np.int64)
    return np.maximum(0, 4000 - 9 * (i % 900) + r.integers(0, 3, n)).astype(np.uint64)  # feet below zero


@pytest.mark.parametrize("m", [64, 127, 128, 129, 131, 256, 300, 1000, 1016, 1100])
@pytest.mark.parametrize("kind", ["noise1", "convex", "edge52", "below52", "mixed", "pow2", "feet"])
def test_boundaries(gpu, kind, m):
    import torch
    n = 64 * m + 3 * m // 2 + 5 if m < 256 else 40 * m + 17
    v = data(kind, n, m)
    st, en = glc.partition(torch.from_numpy(v).cuda(), glc.PART_GPU_SPLITMERGE, m)
    ref = O.compress(v, O.PART_SPLITMERGE_EXACT, m)
    assert np.array_equal(st, ref.start) and np.array_equal(en, ref.end)


@pytest.mark.parametrize("J", [1, 8191, 8192, 8193, 16385])
def test_chain_chunks(gpu, J):
    # starts at the edges of the chain's chunks of 8192 entries
    import torch
    r = np.random.default_rng(J)
    v = (np.arange(4 * J) * 7 + np.cumsum(r.integers(0, 3, 4 * J) * (r.random(4 * J) < 0.02) * 1000)).astype(np.int64)
    st, en = glc.partition(torch.from_numpy(v).cuda(), glc.PART_GPU_SPLITMERGE, 4)
    ref = O.compress(v, O.PART_SPLITMERGE_EXACT, 4)
    assert np.array_equal(st, ref.start) and np.array_equal(en, ref.end)
