"""Fit of mixed partition sizes at both register budgets of 64-bit columns.

Averages of 1024 values and below, above it, of 8192 and above: the rule's edges,
with partitions of each form (a wave's, a workgroup's from registers, two reads) in
every column.  Parameters, widths and payload must equal the oracle's."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [2048, 700, 1024, 1025, 2049, 4096, 8192, 8193, 300]  # the first one: the reduction's block size 256


@pytest.mark.parametrize("pad", [0, 2, 14, 400])
@pytest.mark.parametrize("dt", [np.int64, np.uint64, np.int32])
def test_fit_mixed(gpu, dt, pad):
    import torch
    sizes = SIZES + ([30000, 60000, 50000] if pad == 0 else [256] * pad)
    en = np.cumsum(sizes)
    n = int(en[-1])
    r = np.random.default_rng(pad)
    v = (np.arange(n) * 7 + r.integers(0, 5000, n)).astype(dt)
    st = np.append([0], en[:-1]).astype(np.int32)
    col = glc.compress_partitions(torch.from_numpy(v).cuda(), st, en.astype(np.int32))
    ref = O.compress_parts(v, st, en.astype(np.int32))
    m = col.meta()
    for key in ("model_type", "bits", "bit_offset", "error_bound"):
        assert np.array_equal(m[key], getattr(ref, key)), key
    assert np.array_equal(m["params"].view(np.uint64), ref.params.view(np.uint64))
    assert np.array_equal(col.payload(), ref.words)
