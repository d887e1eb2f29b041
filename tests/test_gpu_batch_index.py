"""The batch's index by one workgroup a column, at its limits.

It is taken up to 2048 partitions and tiles in the largest column and walks 256 of
them at a time: columns of 0, 1, 255, 256, 257, 511, 512, 513 and 2048 partitions,
and with one of 2049 the other path.  Every column must equal the oracle's; twice
over other values in the same buffers, and once from a graph."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [7, 256, 1024, 1500])
@pytest.mark.parametrize("largest", [513, 2048, 2049])
def test_batch_index(gpu, size, largest):
    import torch
    r = np.random.default_rng(size + largest)
    parts = [1, 0, 255, 256, 257, largest, 511, 512]
    dts = [np.int32, np.int64, np.uint32, np.uint64]
    n = [max(0, p * size - (size // 3 if k % 2 else 0)) for k, p in enumerate(parts)]
    dev = [torch.zeros(m, dtype=torch.int32 if k % 2 == 0 else torch.int64, device="cuda").view(
        [torch.int32, torch.int64, torch.uint32, torch.uint64][k % 4]) for k, m in enumerate(n)]
    b = glc.Batch(dev, size)
    outs = [torch.empty_like(t) for t in dev]
    for rep in range(3):
        vals = [(np.arange(m) * 3 + r.integers(0, 1 << (3 + 7 * rep), m)).astype(dts[k % 4]) for k, m in enumerate(n)]
        for t, v in zip(dev, vals):
            t.copy_(torch.from_numpy(v))
        torch.cuda.synchronize()
        if rep < 2:
            b.compress()
            b.decompress(outs)
        else:
            b.run_graph(glc.BATCH_COMPRESS | glc.BATCH_DECOMPRESS, outs)
        torch.cuda.synchronize()
        bits, _ = b.sizes()
        for k, v in enumerate(vals):
            assert np.array_equal(outs[k].cpu().numpy(), v), (rep, k)
            if len(v) == 0:
                assert bits[k] == 0
                continue
            ref = O.compress(v, O.PART_FIXED, size)
            assert bits[k] == ref.total_bits
            m = b.column(k).meta()
            for key in ("start", "end", "model_type", "bits", "bit_offset"):
                assert np.array_equal(m[key], getattr(ref, key)), (rep, k, key)
            assert np.array_equal(b.column(k).payload(), ref.words), (rep, k)
