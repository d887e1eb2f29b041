"""Full decode of columns whose partitions and gaps are whole tiles.

No tile holds more than one partition, so the decode takes the kernels without the
spanning paths; a gap's tiles still go through the search and must come out 0.
Whole numbers, no tolerance."""
import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.int32, np.uint32, np.int64, np.uint64])
def test_gaps(gpu, dt):
    import torch
    n = 40 * 1024 + 77
    st = np.array([0, 1, 3, 4, 9, 9, 20, 38]) * 1024  # gaps, an empty partition, a tail past the last one
    en = np.array([1, 2, 4, 9, 9, 16, 36, 39]) * 1024
    r = np.random.default_rng(3)
    for noise in (1, 300, 1 << 20):
        v = (np.arange(n) * 3 + r.integers(0, noise, n)).astype(dt)
        x = torch.from_numpy(v).cuda()
        col = glc.compress_partitions(x, st.astype(np.int32), en.astype(np.int32))
        want = np.zeros(n, dt)
        for s, e in zip(st, en):
            want[s:e] = v[s:e]
        buf = torch.empty(n + 1, dtype=x.view(torch.int32 if v.itemsize == 4 else torch.int64).dtype, device="cuda")
        for plain in (False, True):
            if plain:
                col.preunpack()
            for sch in (None, glc.DECODE_TILE_W1, glc.DECODE_TILE_W4, glc.DECODE_HALF_TILE_W1):
                if sch is not None:
                    col.set_decode_schedule(sch)
                for mode in (glc.FULL_AUTO, glc.FULL_BITPACKED, glc.FULL_V2):
                    for shift in (0, 1):  # 1: the output is not 16-byte aligned
                        buf.fill_(-1)
                        out = buf[shift:n + shift].view(x.dtype)
                        col.decompress_full(mode, out=out)
                        assert np.array_equal(out.cpu().numpy(), want), (noise, plain, sch, mode, shift)
