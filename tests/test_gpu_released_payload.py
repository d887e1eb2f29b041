"""Packed decodes of columns whose payload holds no bits and was released.

A column of exact lines has fields of 0 bits.  After preunpack(free_packed=True)
its packed modes, schedules and the autotuner still run: they need no payload.
Partitions of one tile, of several tiles, of fewer than four and of more than three
to a tile, and of more than 96; aligned outputs and others.  Values must equal the
column: whole numbers, no tolerance."""
import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [9, 64, 1000, 1024, 4096])
@pytest.mark.parametrize("dt", [np.int32, np.uint32, np.int64, np.uint64])
def test_zero_width_columns(gpu, dt, size):
    import torch
    n = 5 * 4096 + 37
    v = np.full(n, 77, dt)
    col = glc.compress(torch.from_numpy(v).cuda(), glc.PART_FIXED, size)
    assert col.info().total_bits == 0
    col.preunpack(free_packed=True)
    assert not col.info().has_packed
    want = torch.from_numpy(v.view(np.int32 if v.itemsize == 4 else np.int64)).cuda()
    buf = torch.empty(n + 1, dtype=want.dtype, device="cuda")
    for sch in (None, glc.DECODE_TILE_W1, glc.DECODE_TILE_W4, glc.DECODE_HALF_TILE_W1):
        if sch is not None:
            col.set_decode_schedule(sch)
        for shift in (0, 1):  # 1: the output is not 16-byte aligned
            for decode in (lambda o: col.decompress_full(glc.FULL_BITPACKED, out=o),
                           lambda o: col.decompress_full(glc.FULL_AUTO, out=o),
                           lambda o: col.decompress_full_fixed(size, out=o)):
                buf.fill_(-1)
                out = buf[shift:n + shift]
                decode(out)
                assert torch.equal(out, want), (sch, shift)
    col.autotune_decode(buf[:n], reps=1)
    buf.fill_(-1)
    col.decompress_full(glc.FULL_BITPACKED, out=buf[:n])
    assert torch.equal(buf[:n], want)
