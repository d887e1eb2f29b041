"""Lookups in columns whose tiles hold several partitions.

Four lookups of a lane search their partitions together: tiles of 1 to over 90
partitions, empty ones, gaps, elements before the first and after the last
partition, positions outside the column, query counts around a block's 1024, and
column shapes on both sides of the rule for pre-unpacked lookups (8192 values a
partition).  Values must equal the column (0 in gaps): whole numbers, no
tolerance."""
import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


def layout(kind, n, seed):
    r = np.random.default_rng(seed)
    if kind == "runs":  # 0 to 700 values, some gaps, one at both ends
        st, en, at = [], [], 37
        while at < n - 40:
            st.append(at)
            en.append(min(at + int(r.choice([0, 1, 5, 64, 65, 340, 700])), n - 40))
            at = en[-1] + (int(r.integers(1, 90)) if r.random() < 0.1 else 0)
        return np.array(st, np.int32), np.array(en, np.int32)
    if kind == "long":  # two tiles of several partitions, the rest whole ones of one
        st = np.array([0, 20000, 20010, 40500])
        return st.astype(np.int32), np.append(st[1:], n).astype(np.int32)
    cuts = np.unique(np.append(r.integers(0, n, n // int(kind)), [0]))  # no fixed size
    return cuts.astype(np.int32), np.append(cuts[1:], n).astype(np.int32)


@pytest.mark.parametrize("lay", ["runs", "long", "11", "100", "1000"])
@pytest.mark.parametrize("dt", [np.int32, np.uint32, np.int64, np.uint64])
def test_lookups(gpu, dt, lay):
    import torch
    n = 60 * 1024 + 77
    r = np.random.default_rng(n)
    i = np.arange(n, dtype=np.int64)
    wide = (1 << 45) if np.dtype(dt).itemsize == 8 else (1 << 20)
    v = (i * 5 + r.integers(0, wide, n) * (i // 9000 % 2) + r.integers(0, 50, n)).astype(dt)
    st, en = layout(lay, n, 3)
    col = glc.compress_partitions(torch.from_numpy(v).cuda(), st, en)
    want = np.zeros(n, dt)
    for s, e in zip(st, en):
        want[s:e] = v[s:e]
    for q in (1, 1023, 1024, 1025, 20011):
        pos = r.integers(0, n, q)
        pos[::17] = r.choice([-1, -(1 << 31), n, n + 5, (1 << 31) - 1, 0, n - 1], len(pos[::17]))
        ok = (pos >= 0) & (pos < n)
        ref = np.where(ok, want[np.where(ok, pos, 0)], dt(0))
        for pt in (np.int32, np.int64):
            got = col.random_access(torch.from_numpy(pos.astype(pt)).cuda())
            assert np.array_equal(got.cpu().numpy(), ref), (q, pt)
    plain = glc.compress_partitions(torch.from_numpy(v).cuda(), st, en)
    plain.preunpack()
    got = plain.random_access(torch.from_numpy(pos.astype(np.int32)).cuda())
    assert np.array_equal(got.cpu().numpy(), ref)
