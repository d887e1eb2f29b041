"""GPU split/merge where the choice of a block's hull candidates has edges.

Boundaries must equal the oracle's exact-sum split/merge: whole numbers, no
tolerance.  Block sizes: 1, 2 and 3 (ends only, one inner point), 16 and 17 (one row
of anchors and one value more), 63 to 66 (one or two ballots), 113 and 128 (the last
row with one value, a full one), and a last block of every length that leaves.  Data:
exact lines and kinks (every point on a chord), kinks with noise (a second choice of
anchors), steps (ties), products of differences past 2^53 (no certain side), one
value far outside."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def data(kind, n, seed):
    r = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    if kind == "kinks":
        return np.abs(i % 401 - 200) * 1000 + 3
    if kind == "noisy_kinks":
        return np.abs(i % 173 - 86) * 3000 + r.integers(0, 1000, n)
    if kind == "steps":
        return (i // 37) * 1000 + r.integers(0, 2, n)
    if kind == "wide":
        return r.integers(-(1 << 51), 1 << 51, n) // (1 + 4095 * (i // 500 % 2))
    return i * 3 + np.where(r.random(n) < 0.01, 1 << 40, 0)


@pytest.mark.parametrize("m", [1, 2, 3, 16, 17, 63, 64, 65, 66, 113, 128])
@pytest.mark.parametrize("kind", ["kinks", "noisy_kinks", "steps", "wide", "outliers"])
def test_boundaries(gpu, kind, m):
    import torch
    for tail in (0, 1, m // 2, m - 1):
        n = 70 * m + tail
        v = data(kind, n, m + tail)
        st, en = glc.partition(torch.from_numpy(v).cuda(), glc.PART_GPU_SPLITMERGE, m)
        ref = O.compress(v, O.PART_SPLITMERGE_EXACT, m)
        assert np.array_equal(st, ref.start) and np.array_equal(en, ref.end)
