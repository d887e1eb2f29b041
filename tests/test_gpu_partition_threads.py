"""V6 and split/merge encodes from several threads on streams of their own.

The partitioners' device scratch is shared: a call's boundaries must be copied out of
it before the next call's kernels, on another stream, write it, also where the next
column is larger and the scratch is replaced.  Blobs must equal those of calls one at a
time: bytes, no tolerance."""
import threading

import numpy as np
import pytest

import glc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("part,size,base", [(glc.PART_V6, 0, 256), (glc.PART_GPU_SPLITMERGE, 64, 0)])
def test_streams(gpu, part, size, base):
    import torch
    sizes = [3000, 700_000, 40_000, 90_001, 1 << 20, 5000]
    cols = [torch.from_numpy(np.cumsum(np.random.default_rng(k).integers(0, 99, n)).astype(np.int64)).cuda()
            for k, n in enumerate(sizes)]
    torch.cuda.synchronize()
    want = [glc.compress(x, part, size, base).serialize() for x in cols]
    bad = []

    def work(order):
        try:
            s = torch.cuda.Stream()
            for _ in range(8):
                for k in order:
                    if glc.compress(cols[k], part, size, base, stream=s).serialize(stream=s) != want[k]:
                        bad.append(k)
        except Exception as e:
            bad.append(e)

    ts = [threading.Thread(target=work, args=(o,)) for o in ((0, 1, 2, 3, 4, 5), (5, 4, 3, 2, 1, 0), (2, 4, 0, 5, 1, 3))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
