"""Full decode into outputs that are not 16-byte aligned.

Their rows are cut at the output's 128-byte lines, so every offset from a line
counts: all of them, for whole tiles of each extraction form (up to 32 bits, wider,
DIRECT_COPY, pre-unpacked), tiles of few and of many partitions and more than the
staged map holds, and columns that end before, in and after a tile's last row.  Values
must equal the column and nothing beside the output may change: whole numbers."""
import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


def column(dt, kind, n):
    r = np.random.default_rng(n)
    i = np.arange(n, dtype=np.int64)
    if kind == "narrow":
        return (i * 3 + r.integers(0, 500, n)).astype(dt)
    if np.dtype(dt).itemsize == 4:  # residuals of up to 33 bits
        return r.integers(np.iinfo(dt).min, np.iinfo(dt).max, n, endpoint=True).astype(dt)
    if kind == "far":
        return ((1 << 58) + i * 1000 + r.integers(0, 1 << 18, n)).astype(dt)  # uint64: DIRECT_COPY
    return (i * 11 + r.integers(0, 1 << 45, n)).astype(dt)


@pytest.mark.parametrize("size", [9, 64, 700, 1024, 3000])
@pytest.mark.parametrize("dt", [np.int32, np.uint32, np.int64, np.uint64])
def test_every_offset_from_a_line(gpu, dt, size):
    import torch
    k = 128 // np.dtype(dt).itemsize
    signed = {4: torch.int32, 8: torch.int64}[np.dtype(dt).itemsize]
    for kind, tail in (("narrow", 1), ("wide", 1023), ("far", 995)):
        n = 4 * 1024 + tail
        v = column(dt, kind, n)
        x = torch.from_numpy(v).cuda()
        col = glc.compress(x, glc.PART_FIXED, size)
        buf = torch.empty(n + 2 * k, dtype=signed, device="cuda")
        assert buf.data_ptr() % 128 == 0
        want = x.view(signed)
        for plain in (False, True):
            if plain:
                col.preunpack()
            for sch in (glc.DECODE_TILE_W1, glc.DECODE_TILE_W4, glc.DECODE_HALF_TILE_W1):
                col.set_decode_schedule(sch)
                for shift in range(1, k + 1):
                    buf.fill_(-1)
                    col.decompress_full(glc.FULL_AUTO, out=buf[shift:shift + n])
                    assert torch.equal(buf[shift:shift + n], want), (kind, plain, sch, shift)
                    assert int((buf[:shift] != -1).sum()) == 0 and int((buf[shift + n:] != -1).sum()) == 0
