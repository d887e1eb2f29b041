"""Columns around the sizes where one workgroup stops doing a whole step.

The index of up to 4096 partitions and 4096 tiles is one launch, V6 thresholds and
partitions of up to 2048 blocks another, more take the long forms: metadata, payload,
blob and decode must equal the oracle's on both sides, also where the two limits
disagree, after a round trip through the blob, and from two threads at once."""
import threading

import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def check(v, part, opart, size=0, base=0):
    import torch
    col = glc.compress(torch.from_numpy(v).cuda(), part, size, base)
    ref = O.compress(v, opart, base_size=base) if base else O.compress(v, opart, size)
    m = col.meta()
    for k, r in [("start", ref.start), ("end", ref.end), ("model_type", ref.model_type), ("bits", ref.bits),
                 ("bit_offset", ref.bit_offset), ("error_bound", ref.error_bound)]:
        assert np.array_equal(m[k], r), k
    assert np.array_equal(m["params"].view(np.uint64), ref.params.view(np.uint64))
    assert np.array_equal(col.payload(), ref.words)
    blob = col.serialize()
    assert blob == ref.blob
    back = glc.deserialize(blob, col.dtype)
    pos = torch.from_numpy(np.arange(0, v.size, 37, dtype=np.int32)).cuda()
    for c in (col, back):
        assert np.array_equal(c.decompress_full().cpu().numpy(), v)
        assert np.array_equal(c.random_access(pos).cpu().numpy(), v[::37])


def ramp(n, dt, seed):
    r = np.random.default_rng(seed)
    return (np.arange(n) * 3 + r.integers(0, 1 + (1 << (seed % 9)), n)).astype(dt)


@pytest.mark.parametrize("P", [1, 1023, 1024, 1025, 4095, 4096, 4097])
@pytest.mark.parametrize("S", [16, 300])
def test_partitions_around_one_workgroup(gpu, P, S):
    check(ramp(P * S - 5, np.int64, P), glc.PART_FIXED, O.PART_FIXED, S)


@pytest.mark.parametrize("tiles", [4095, 4096, 4097])
def test_tiles_around_one_workgroup(gpu, tiles):
    check(ramp(tiles * 1024 - 7, np.uint32, tiles), glc.PART_FIXED, O.PART_FIXED, 8192)


@pytest.mark.parametrize("blocks", [1, 2, 1024, 1025, 2047, 2048, 2049, 16384, 16385])
def test_v6_blocks_around_one_workgroup(gpu, blocks):
    r = np.random.default_rng(blocks)
    n = blocks * 32 - 3  # base 4: blocks of 32 values
    v = np.cumsum(r.integers(0, 1 + r.integers(1, 50, n), n)).astype(np.uint64)
    check(v, glc.PART_V6, O.PART_V6, base=4)


def test_v6_from_two_threads(gpu):
    import torch
    cols = [torch.from_numpy(np.cumsum(np.random.default_rng(k).integers(0, 99, n)).astype(np.int64)).cuda()
            for k, n in enumerate((5000, 300_000, 40_000))]
    want = [glc.compress(x, glc.PART_V6).serialize() for x in cols]
    bad = []

    def work(order):
        try:
            for _ in range(5):
                for k in order:
                    if glc.compress(cols[k], glc.PART_V6).serialize() != want[k]:
                        bad.append(k)
        except Exception as e:
            bad.append(e)

    ts = [threading.Thread(target=work, args=(o,)) for o in ((0, 1, 2), (2, 1, 0))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
