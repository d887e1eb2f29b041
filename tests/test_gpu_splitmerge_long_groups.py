"""GPU split/merge groups of many candidates: those left open by the growth of all
starts at once and completed on the walk.

Small minimum sizes on smooth data (over a thousand candidates a group), values all
near 0 (one group for the whole column), columns where such stretches alternate with
short groups, and values beyond 2^52 (read, not bounded by hulls).  Boundaries must
equal the oracle's: whole numbers, no tolerance."""
import time

import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def data(kind, n):
    r = np.random.default_rng(n)
    i = np.arange(n, dtype=np.int64)
    if kind == "line":
        return (i * 5 + 3).astype(np.int32)
    if kind == "slope":
        return np.floor(i * 0.37).astype(np.uint32)
    if kind == "zeros":
        return np.zeros(n, np.int64)
    if kind == "flags":
        return r.integers(0, 2, n).astype(np.uint64)
    if kind == "far":
        return ((1 << 60) + i * 977).astype(np.int64)
    stretch = (i // 20000) % 2  # lines, and short runs at random offsets
    return np.where(stretch == 0, i * 7, r.integers(0, 1 << 40, n // 60 + 1)[i // 60] + (i % 60) * 3).astype(np.int64)


@pytest.mark.parametrize("m", [1, 2, 5, 16])
@pytest.mark.parametrize("kind", ["line", "slope", "zeros", "flags", "far", "alternating"])
def test_boundaries(gpu, kind, m):
    import torch
    n = 100_003 if m < 5 else 150_001
    v = data(kind, n)
    st, en = glc.partition(torch.from_numpy(v).cuda(), glc.PART_GPU_SPLITMERGE, m)
    ref = O.compress(v, O.PART_SPLITMERGE_EXACT, m)
    assert np.array_equal(st, ref.start) and np.array_equal(en, ref.end)


def test_one_group_for_a_long_column(gpu):
    # 18079 starts, each of whose groups would take in the rest of 2^26 values: 4e11
    # steps of a wave if all were grown to the end, over a minute at the whole GPU's
    # pace of about 3 to the nanosecond; 7e7 steps, 25 ms, on the walk alone
    import torch
    x = torch.zeros(1 << 26, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    t = time.perf_counter()
    st, en = glc.partition(x, glc.PART_GPU_SPLITMERGE, 128)
    torch.cuda.synchronize()
    took = time.perf_counter() - t
    assert st.tolist() == [0] and en.tolist() == [1 << 26]
    assert took < 5.0
