"""The fit's forms at their edges: theta bits, widths, offsets and payload equal the oracle's.

Lengths around what a wave (1024, 2048) and a workgroup (4096, 8192) hold, above
it, and around 2^17, where the index sums stop being taken in closed form; values
around 2^51, 2^52 and 2^53 (the exact FP64 residual, the conversion constant,
DIRECT_COPY) and nanosecond timestamps; block sizes other than 256 over short and long
partitions (the first partition sets it).  Bits and whole numbers: no tolerance."""
import numpy as np
import pytest

import glc
import oracle as O

pytestmark = pytest.mark.gpu


def same(col, ref):
    m = col.meta()
    for k, r in [("start", ref.start), ("end", ref.end), ("model_type", ref.model_type), ("bits", ref.bits),
                 ("bit_offset", ref.bit_offset), ("error_bound", ref.error_bound)]:
        assert np.array_equal(m[k], r), k
    assert np.array_equal(m["params"].view(np.uint64), ref.params.view(np.uint64)), "theta bits"
    assert np.array_equal(col.payload(), ref.words), "payload"


def values(kind, n, seed):
    r = np.random.default_rng(seed)
    i = np.arange(n, dtype=np.int64)
    return {"i32": lambda: (i * 5 % (1 << 30) + r.integers(-300, 300, n)).astype(np.int32),
            "u32": lambda: (i * 3 % (1 << 31) + r.integers(0, 1 << 12, n)).astype(np.uint32),
            "i64": lambda: (i * 1000 + r.integers(-5000, 5000, n)).astype(np.int64),
            "2^51": lambda: ((1 << 51) - 4 * n + i * 4 + r.integers(-9, 9, n)).astype(np.int64),
            "-2^52": lambda: (-(1 << 52) + i - r.integers(0, 3, n)).astype(np.int64),
            "2^53": lambda: ((1 << 53) - 8 + (i % 700) * (i % 3 == 0) // 40).astype(np.uint64),
            "ns": lambda: (1_700_000_000_000_000_000 + np.cumsum(r.integers(0, 2000, n))).astype(np.int64),
            "u64": lambda: ((1 << 40) + i * 77 + r.integers(0, 1 << 20, n)).astype(np.uint64)}[kind]()


@pytest.mark.parametrize("kind", ["i32", "u32", "i64", "2^51", "-2^52", "2^53", "ns", "u64"])
def test_explicit_lengths(gpu, kind):
    import torch
    lens = [256, 257, 1000, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 3, 0, 20000]
    en = np.cumsum(lens).astype(np.int32)
    st = (en - lens).astype(np.int32)
    v = values(kind, int(en[-1]), len(kind))
    same(glc.compress_partitions(torch.from_numpy(v).cuda(), st, en), O.compress_parts(v, st, en))


@pytest.mark.parametrize("S", [224, 225, 256, 1024, 1025, 2047, 2048, 4096, 4097, 8192, 8193])
@pytest.mark.parametrize("kind", ["i32", "2^51", "2^53", "ns"])
def test_fixed_sizes(gpu, kind, S):
    import torch
    v = values(kind, 5 * S + 13, S)
    same(glc.compress(torch.from_numpy(v).cuda(), glc.PART_FIXED, S), O.compress(v, O.PART_FIXED, S))


@pytest.mark.parametrize("first", [1, 32, 33, 96, 128, 200, 224])
def test_other_block_sizes(gpu, first):
    import torch
    lens = [first, 5, 64, 900, 1024, 1025, 3000, 9000]
    en = np.cumsum(lens).astype(np.int32)
    st = (en - lens).astype(np.int32)
    for kind in ("u32", "i64", "2^53"):
        v = values(kind, int(en[-1]), first)
        same(glc.compress_partitions(torch.from_numpy(v).cuda(), st, en), O.compress_parts(v, st, en))


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17, (1 << 17) + 1, 400_000])
def test_long_partitions(gpu, n):
    import torch
    v = values("i64", n, n % 97)
    same(glc.compress(torch.from_numpy(v).cuda(), glc.PART_FIXED, n), O.compress(v, O.PART_FIXED, n))
    for S in (1024, 2048, 5000):
        b = glc.Batch([torch.from_numpy(v).cuda(), torch.from_numpy(v[:100]).cuda()], S)
        b.compress()
        same(b.column(0), O.compress(v, O.PART_FIXED, S))
        same(b.column(1), O.compress(v[:100], O.PART_FIXED, S))
    b = glc.Batch([torch.from_numpy(v).cuda()], n)
    b.compress()
    same(b.column(0), O.compress(v, O.PART_FIXED, n))
