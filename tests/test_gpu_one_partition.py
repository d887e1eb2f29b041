"""One partition of nearly 2^31 values: every loop over a partition's values ends
where an index past the last one would no longer be an int32.

A fixed partition (a workgroup, block size 256), an explicit list whose short
first partition sets a block size below 256, and a batch (a wave).  The decoded
values must equal the column: whole numbers, no tolerance."""
import pytest
import torch

import glc

pytestmark = [pytest.mark.gpu, pytest.mark.slow]

NMAX = (1 << 31) - 1


@pytest.fixture(scope="module")
def column(gpu):
    print(f"generate {NMAX} int32 values on the GPU", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(41)
    x = torch.arange(NMAX, device="cuda", dtype=torch.int32) >> 1
    x += torch.randint(-4096, 4097, (NMAX,), generator=g, device="cuda", dtype=torch.int32)
    return x, torch.empty_like(x)


def check(col, x, out, p):
    m = col.meta()
    assert m["end"][p] == NMAX and m["error_bound"][p] >= 4096
    out.fill_(-1)
    col.decompress_full(glc.FULL_BITPACKED, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out, x)


def test_fixed(column):
    x, out = column
    check(glc.compress(x, glc.PART_FIXED, NMAX), x, out, 0)


def test_after_a_short_one(column):
    import numpy as np
    x, out = column
    print("block size below 256", flush=True)
    check(glc.compress_partitions(x, np.array([0, 200], np.int32), np.array([200, NMAX], np.int32)), x, out, 1)


def test_batch(column):
    x, out = column
    print("batch", flush=True)
    b = glc.Batch([x], NMAX)
    b.compress()
    torch.cuda.synchronize()
    check(b.column(0), x, out, 0)
    del b
