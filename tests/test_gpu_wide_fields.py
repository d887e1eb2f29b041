"""Full decode of 33- to 64-bit fields by half tiles and across partitions.

Two such fields of a lane come from five words, wherever the first one starts in
its word, and a half tile holds half of a wide tile's rows.  Widths at the ends of
the range and around 48, partition sizes that leave every kind of tile (whole, two
and three partitions), and columns that end in either half of the last tile.
Values must equal the column: whole numbers, no tolerance."""
import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [401, 500, 777, 1000, 1024, 1500, 4096])
@pytest.mark.parametrize("bits", [33, 34, 47, 48, 49, 62, 63, 64])
def test_wide_fields(gpu, bits, size):
    import torch
    for k, dt in enumerate((np.int64, np.uint64)):
        r = np.random.default_rng(bits * 10 + k)
        n = 12 * 1024 + [1, 600][k] + 4096 * (bits % 2)
        v = r.integers(0, (1 << bits) - 1, n, dtype=np.uint64, endpoint=True)
        v = (v >> np.uint64(1)).astype(dt) if bits < 64 else v.astype(dt)  # a sign bit more
        x = torch.from_numpy(v).cuda()
        col = glc.compress(x, glc.PART_FIXED, size)
        for sch in (None, glc.DECODE_TILE_W1, glc.DECODE_TILE_W4, glc.DECODE_HALF_TILE_W1):
            if sch is not None:
                col.set_decode_schedule(sch)
            for mode in (glc.FULL_BITPACKED, glc.FULL_V2):
                assert np.array_equal(col.decompress_full(mode).cpu().numpy(), v), (dt, sch, mode)
        col.preunpack()
        assert np.array_equal(col.decompress_full(glc.FULL_PREUNPACKED).cpu().numpy(), v)
