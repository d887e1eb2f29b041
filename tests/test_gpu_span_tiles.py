"""Full decode of 1024-value tiles that hold several partitions.

Three paths by the partitions a tile touches: up to three (a wave per partition
in turn), up to 96 (the staged map), more or a shared start (the search).  Sizes at
those edges, tails, gaps, empty partitions, first partition after the column's
start, widths of each extraction form (0, <= 16, <= 32, > 32 bits, DIRECT_COPY,
64-bit predictions beyond 2^50) and outputs that are not 16-byte aligned.  Values
must equal the column (0 in gaps): whole numbers, no tolerance."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def column(dt, kind, n, seed):
    r = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    if kind == "narrow":
        return (i * 3 + r.integers(0, 500, n)).astype(dt)
    if kind == "mid":
        return (i * 7 + r.integers(0, 1 << 22, n)).astype(dt)
    if kind == "const":
        return np.full(n, 77, dt)
    if np.dtype(dt).itemsize == 4:  # residuals of up to 33 bits
        return r.integers(np.iinfo(dt).min, np.iinfo(dt).max, n, endpoint=True).astype(dt)
    if kind == "far":
        return ((1 << 58) + i * 1000 + r.integers(0, 1 << 18, n)).astype(dt)  # uint64: DIRECT_COPY
    return (i * 11 + r.integers(0, 1 << 45, n)).astype(dt)


def layout(kind, n, seed):
    r = np.random.default_rng(seed)
    if kind == "runs":  # 1 to 700 values, some empty, some gaps, a gap at both ends
        st, en, at = [], [], 37
        while at < n - 40:
            ln = int(r.choice([0, 1, 5, 11, 63, 64, 65, 200, 340, 341, 700]))
            st.append(at)
            en.append(min(at + ln, n - 40))
            at = en[-1] + (int(r.integers(1, 90)) if r.random() < 0.1 else 0)
        return np.array(st, np.int32), np.array(en, np.int32)
    size = int(kind)
    st = np.arange(0, n, size)
    return st.astype(np.int32), np.minimum(st + size, n).astype(np.int32)


LAYOUTS = ["runs", "10", "11", "64", "341", "342", "512", "513", "1000", "1023", "1025", "3000"]


@pytest.mark.parametrize("lay", LAYOUTS)
@pytest.mark.parametrize("dt", [np.int32, np.uint32, np.int64, np.uint64])
def test_decode_spanning_tiles(gpu, dt, lay):
    import torch
    for k, kind in enumerate(["narrow", "mid", "const", "far", "wide"]):
        n = 9 * 1024 + [0, 1, 511, 1023, 77][k]
        v = column(dt, kind, n, k)
        st, en = layout(lay, n, k)
        x = torch.from_numpy(v).cuda()
        col = glc.compress_partitions(x, st, en)
        want = np.zeros(n, dt)
        for s, e in zip(st, en):
            want[s:e] = v[s:e]
        signed = {4: torch.int32, 8: torch.int64}[v.itemsize]
        modes = [glc.FULL_BITPACKED, glc.FULL_WORKSTEAL]
        for plain in (False, True):
            if plain:
                col.preunpack()
                modes = [glc.FULL_PREUNPACKED]
            for mode in modes:
                for sch in (glc.DECODE_TILE_W1, glc.DECODE_TILE_W4, glc.DECODE_HALF_TILE_W1):
                    col.set_decode_schedule(sch)
                    for shift in (0, 1):  # 1: the output is not 16-byte aligned
                        buf = torch.full((n + 1,), -1, dtype=signed, device="cuda")
                        out = buf[shift:n + shift].view(x.dtype)
                        col.decompress_full(mode, out=out)
                        got = out.cpu().numpy()
                        assert np.array_equal(got, want), (kind, mode, sch, shift)
                        assert int(buf[n if shift == 0 else 0]) == -1  # nothing beside the output
        ref = O.compress_parts(v, st, en)
        assert np.array_equal(col.payload(), ref.words)


def test_batch_spanning_tiles(gpu):
    import torch
    cols = [column(dt, kind, n, 5) for dt in (np.int32, np.uint32, np.int64, np.uint64)
            for kind, n in (("narrow", 1), ("mid", 1023), ("far", 5000), ("wide", 3 * 1024 + 1))]
    for size in (9, 64, 300, 1000, 1025):
        b = glc.Batch([torch.from_numpy(c).cuda() for c in cols], size)
        b.compress()
        for w, t in glc.BATCH_SCHEDULES:
            b.set_schedule(w, t)
            for o, c in zip(b.decompress(), cols):
                assert np.array_equal(o.cpu().numpy(), c), (size, w, t, c.dtype, c.size)
