"""What a program does with this framework, as cases that can be timed.

A case is one call (or the calls that belong together) on a column:

  compress  encode a device column: glc.compress
  decode    decode a whole column: Column.decompress_full
  lookup    random access: Column.random_access
  batch     many columns encoded and decoded by one recorded graph: glc.Batch
  blob      store and load: serialize, deserialize, decode

Columns are synthetic, made on the GPU from the seed: `linear` (a ramp with
uniform noise that takes noise + 1 bits), `segments` (piecewise linear, glc.workloads) and
`sorted` (keys with exponential gaps and 1 % bursts, like timestamps).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "g-leco_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import glc  # noqa: E402
from glc import workloads  # noqa: E402

PARTITIONERS = {"fixed": glc.PART_FIXED, "v6": glc.PART_V6, "splitmerge": glc.PART_GPU_SPLITMERGE}
DTYPES = {"i32": glc.I32, "u32": glc.U32, "i64": glc.I64, "u64": glc.U64}
MODES = {"auto": glc.FULL_AUTO, "v2": glc.FULL_V2, "steal_adv": glc.FULL_WORKSTEAL_ADV}


def listed():
    return [
        # the smallest calls: 10^5 lookups in, a decode and an encode of a
        # column of a few MB, where launches and host work count
        dict(name="lookup_small", kind="lookup", data="linear", noise=6, dtype="i32", n=1 << 20, part="fixed",
             size=1024, q=100_000, plain=False),
        dict(name="decode_small", kind="decode", data="linear", noise=6, dtype="i32", n=1 << 20, part="fixed",
             size=1024, mode="auto", plain=False),
        dict(name="compress_small", kind="compress", data="linear", noise=6, dtype="i32", n=65_537, part="fixed",
             size=1024),
        # the main workload: a 2 GiB uint64 column of piecewise-linear keys,
        # variable partitions; encode, full scan, and half-uniform half-Zipf lookups
        dict(name="compress_v6", kind="compress", data="segments", dtype="u64", n=1 << 28, part="v6", size=2048),
        dict(name="decode_v6", kind="decode", data="segments", dtype="u64", n=1 << 28, part="v6", size=2048,
             mode="auto", plain=False),
        dict(name="lookup_v6", kind="lookup", data="segments", dtype="u64", n=1 << 28, part="v6", size=2048,
             q=1 << 24, plain=False),
        # a scan of a timestamp column in the default fixed layout
        dict(name="decode_fixed", kind="decode", data="sorted", dtype="i64", n=300_000_001, part="fixed", size=4096,
             mode="auto", plain=False),
        # partition sizes that a program picks without regard to the tile:
        # a 32-bit id column scanned, a timestamp column encoded
        dict(name="decode_ragged", kind="decode", data="linear", noise=10, dtype="u32", n=50_000_003, part="fixed",
             size=1000, mode="auto", plain=False),
        dict(name="compress_ragged", kind="compress", data="sorted", dtype="i64", n=20_000_003, part="fixed",
             size=1000),
        # the smallest output: cost-driven split/merge partitions, for columns written once
        dict(name="compress_splitmerge", kind="compress", data="segments", dtype="u64", n=1 << 26,
             part="splitmerge", size=128),
        # a table of many columns of mixed type and length, as one graph
        dict(name="batch_mixed", kind="batch", columns=1000, total=1 << 26, size=1024),
        # store and load through the file format
        dict(name="blob_roundtrip", kind="blob", data="linear", noise=18, dtype="i64", n=(1 << 24) + 1000,
             part="fixed", size=4096),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layout(rng, n_max):
    """A column and its partitioning; sizes over their logarithm, mostly odd."""
    c = {"data": rng.choice(["linear", "segments", "sorted"])}
    c["dtype"] = rng.choice(["i64", "u64"] if c["data"] == "segments" else ["i32", "u32", "i64", "u64"])
    if c["data"] == "linear":
        c["noise"] = rng.randint(0, 16 if c["dtype"] in ("i32", "u32") else 36)
    c["n"] = _log_uniform(rng, 4096, n_max)
    c["part"] = rng.choice(["fixed", "fixed", "v6", "splitmerge"])
    if c["part"] == "splitmerge":
        c["n"] = min(c["n"], _log_uniform(rng, 1 << 14, 1 << 25))
        c["size"] = rng.choice([64, 100, 128, 256])
    elif c["part"] == "v6":
        c["size"] = rng.choice([512, 1024, 2048, 4096])
    else:
        c["size"] = rng.choice([256, 512, 1024, 2048, 4096, 8192, _log_uniform(rng, 200, 10_000)])
    return c


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "compress", "compress", "lookup", "lookup", "batch", "blob"])
    if kind == "batch":
        return {"kind": kind, "columns": _log_uniform(rng, 4, 1000), "total": _log_uniform(rng, 1 << 18, 1 << 26),
                "size": rng.choice([512, 1000, 1024, 2048, 4096])}
    c = {"kind": kind, **_layout(rng, {"blob": 1 << 24}.get(kind, 1 << 27))}
    if kind == "blob":  # a blob has the same size for every seed: even noise, no last partition of a few values
        c.update(data="linear", noise=rng.randint(4, 16 if c["dtype"] in ("i32", "u32") else 36), part="fixed",
                 size=max(c["size"], 256))
        c["n"] += 64 if 0 < c["n"] % c["size"] < 64 else 0
    if kind == "decode":
        c["mode"] = rng.choice(["auto", "auto", "auto", "auto", "v2", "steal_adv"])
    if kind == "lookup":
        c["q"] = _log_uniform(rng, 256, 1 << 23)
    if kind in ("decode", "lookup"):
        c["plain"] = rng.random() < 0.2
    return c


# ---- inputs -------------------------------------------------------------------
def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1_000_003 + stream) % (1 << 62))
    return g


def _as_dtype(v, dtype):
    """int64 values as a tensor of the case's element type."""
    if dtype in ("i32", "u32"):
        v = v.to(torch.int32)
        return v.view(torch.uint32) if dtype == "u32" else v
    return v.view(torch.uint64) if dtype == "u64" else v


def _signed(t):
    """The same bits as a signed tensor."""
    return t.view({torch.uint32: torch.int32, torch.uint64: torch.int64}.get(t.dtype, t.dtype))


def _linear(n, noise, narrow, g):
    """floor(m i) + U[-a, a], a = 3/4 of 2^noise, shifted to stay positive; m from the generator."""
    amp = max(1, (3 << noise) >> 2)
    top = min(1 << 10, ((1 << 31) - (1 << 22)) / (n + 1)) if narrow else 1 << 20
    m = float(torch.rand(1, generator=g, device="cuda", dtype=torch.float64)) * (top - top / 64) + top / 64
    v = torch.floor(torch.arange(n, device="cuda", dtype=torch.float64) * m).to(torch.int64)
    v += torch.randint(-amp, amp + 1, (n,), generator=g, device="cuda", dtype=torch.int64)
    v += amp
    return v


def _sorted(n, narrow, g):
    """Sorted keys: exponential gaps, 1 % bursts of 1000 times the mean gap; 64-bit keys are microsecond times."""
    mean = max(1.0, min(1000.0, (1 << 30) / (11.0 * n))) if narrow else 1000.0
    burst = min(1000.0 * mean, (1 << 30) / (0.02 * n)) if narrow else 1000.0 * mean
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    gaps = torch.floor(-mean * torch.log1p(-u)).to(torch.int64)
    gaps[torch.rand(n, generator=g, device="cuda", dtype=torch.float32) < 0.01] = int(burst)
    v = torch.cumsum(gaps, 0)
    if not narrow:
        v += 1_700_000_000_000_000
    return v


def _values(case, seed):
    n, dtype = case["n"], case["dtype"]
    narrow = dtype in ("i32", "u32")
    if case["data"] == "segments":
        v = workloads.c2_uint64_torch(n, seed=int(seed), nseg=max(1, n >> 16)).view(torch.int64)
    elif case["data"] == "sorted":
        v = _sorted(n, narrow, _generator(seed, 1))
    else:
        v = _linear(n, case["noise"], narrow, _generator(seed, 2))
    return _as_dtype(v, dtype)


def _positions(case, seed):
    """Half uniform, half Zipf(1.1) ranks scattered over the column; int32."""
    n, q = case["n"], case["q"]
    g = _generator(seed, 3)
    u = torch.rand(q, generator=g, device="cuda", dtype=torch.float64)
    uniform = (u * n).to(torch.int64)
    rank = (1.0 - u * (1.0 - float(n + 1) ** -0.1)).pow(-10.0).to(torch.int64) - 1
    hot = rank.clamp_(0, n - 1) * 2654435761 % n
    pick = torch.rand(q, generator=g, device="cuda") < 0.5
    return torch.where(pick, uniform, hot).clamp_(0, n - 1).to(torch.int32)


def _batch_lengths(case):
    """Column lengths, log-uniform over [2^10, 2^24] scaled to the total; the same for every seed."""
    r = np.random.default_rng([case["columns"], case["total"]])
    raw = np.exp(r.uniform(math.log(1 << 10), math.log(1 << 24), case["columns"]))
    return [max(64, int(x)) for x in raw * (case["total"] / raw.sum())], r.random(case["columns"]) < 0.5


def _batch_columns(case, seed):
    lens, wide = _batch_lengths(case)
    noise = np.random.default_rng([int(seed) % (1 << 32), 5]).integers(0, 21, len(lens))
    g = _generator(seed, 4)
    cols = []
    for n, w, k in zip(lens, wide, noise):
        v = _linear(n, int(min(k, 20)), not w, g)
        cols.append(v if w else v.to(torch.int32))
    return cols


def _batch_outputs(case):
    """One buffer per element type and each column's part of it, 512-byte aligned as separate tensors would be."""
    lens, wide = _batch_lengths(case)
    total = {False: 0, True: 0}
    at = []
    for n, w in zip(lens, wide):
        at.append(total[bool(w)])
        total[bool(w)] += (n + 127) // 128 * 128
    buffers = {w: torch.zeros(max(total[w], 1), dtype=torch.int64 if w else torch.int32, device="cuda") for w in total}
    parts = [buffers[bool(w)][o:o + n] for n, w, o in zip(lens, wide, at)]
    return buffers, parts


def _compress(values, case):
    size = case["size"]
    return glc.compress(values, PARTITIONERS[case["part"]], 0 if case["part"] == "v6" else size,
                        size if case["part"] == "v6" else 0)


def _archive(case):
    """Device buffers that a compressed column is appended to: its payload and, where the number of partitions
    is the partitioner's choice, its metadata too (None: read in place)."""
    n, size = case["n"], case["size"]
    words = torch.zeros(n * (1 if case["dtype"] in ("i32", "u32") else 2) + 64, dtype=torch.int32, device="cuda")
    if case["part"] == "fixed":
        return [None] * 7 + [words]
    p = -(-n // (8 * size)) * 16 if case["part"] == "v6" else -(-n // size)
    kinds = [torch.int32, torch.int32, torch.int32, torch.float64, torch.int32, torch.int64, torch.int64]
    return [torch.zeros(4 * p if k == torch.float64 else p, dtype=k, device="cuda") for k in kinds] + [words]


def _append(archive, part):
    archive[:part.numel()].copy_(part)
    return archive


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        cols = _batch_columns(case, seed)
        buffers, parts = _batch_outputs(case)
        batch = glc.Batch(cols, case["size"])
        batch.set_outputs(parts)
        return {"kind": kind, "batch": batch, "buffers": [buffers[False], buffers[True]], "parts": parts}
    values = _values(case, seed)
    if kind == "compress":
        return {"kind": kind, "values": values, "case": dict(case), "column": None, "archive": _archive(case)}
    column = _compress(values, case)
    s = {"kind": kind, "column": column, "dtype": DTYPES[case["dtype"]]}
    if case.get("plain"):
        column.preunpack()
    if kind == "lookup":
        s["pos"] = _positions(case, seed)
        s["out"] = torch.empty(case["q"], dtype=values.dtype, device="cuda")
    else:
        s["out"] = torch.empty_like(values)
        s["mode"] = MODES[case.get("mode", "auto")]
    return s


# ---- passes -------------------------------------------------------------------
class _Arrays(ctypes.Structure):  # glc_column_arrays
    _fields_ = [(k, ctypes.c_void_p) for k in ("start", "end", "type", "params", "bits", "offsets", "bounds", "words",
                                               "plain")]


class _View:
    """Device memory of a column as torch takes it."""

    def __init__(self, ptr, count, kind):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": kind, "data": (ptr, False), "version": 2}


def _column_arrays(column):
    """The compressed column's arrays in device memory, as tensors over the column's own memory."""
    a, info = _Arrays(), column.info()
    if glc.lib().glc_column_arrays_get(column.handle, ctypes.byref(a)):
        raise RuntimeError("glc_column_arrays_get failed")
    p = info.num_partitions
    shapes = [(a.start, p, "<i4"), (a.end, p, "<i4"), (a.type, p, "<i4"), (a.params, 4 * p, "<f8"),
              (a.bits, p, "<i4"), (a.offsets, p, "<i8"), (a.bounds, p, "<i8"), (a.words, info.payload_words, "<i4")]
    return [torch.as_tensor(_View(*x), device="cuda") for x in shapes]


def run(state):
    kind = state["kind"]
    if kind == "decode":
        return _signed(state["column"].decompress_full(state["mode"], out=state["out"]))
    if kind == "lookup":
        return _signed(state["column"].random_access(state["pos"], out=state["out"]))
    if kind == "compress":
        state["column"] = None  # the last pass's column is given back first
        state["column"] = _compress(state["values"], state["case"])
        return [x if a is None else _append(a, x)
                for a, x in zip(state["archive"], _column_arrays(state["column"]))]
    if kind == "batch":
        state["batch"].run_graph(glc.BATCH_COMPRESS | glc.BATCH_DECOMPRESS)
        return state["buffers"]
    blob = state["column"].serialize(gpu=True)
    loaded = glc.deserialize(blob, state["dtype"])
    out = _signed(loaded.decompress_full(out=state["out"]))
    loaded.close()
    return [np.frombuffer(blob, np.uint8), out]


# ---- what a pass is held against ------------------------------------------------
def _bits(case):
    """About how many bits a value's residual takes."""
    if case["data"] == "segments":
        return 11.0
    if case["data"] == "linear":
        return case["noise"] + 2.0
    return 12.0 if case["dtype"] in ("i32", "u32") else 19.0


def work(case):
    """Bytes of a pass: values in or out, the packed residuals, 64 bytes per partition."""
    if case["kind"] == "batch":
        lens, wide = _batch_lengths(case)
        raw = sum(n * (8 if w else 4) for n, w in zip(lens, wide))
        packed = sum(n for n in lens) * 12.0 / 8
        return {"bytes": 2 * (raw + packed), "flops": 0}
    n, w = case["n"], 4 if case["dtype"] in ("i32", "u32") else 8
    residual = 8.0 if case.get("plain") else _bits(case) / 8
    if case["kind"] == "lookup":
        return {"bytes": case["q"] * (4 + w + math.ceil(residual)), "flops": 0}
    parts = n / {"fixed": case["size"], "v6": case["size"], "splitmerge": 4096}[case["part"]]
    one = n * (w + residual) + 64.0 * parts
    if case["kind"] == "blob":  # read once and written once as a blob, read again to decode
        return {"bytes": 2 * (n * residual + 64.0 * parts) + one, "flops": 0}
    return {"bytes": one, "flops": 0}


def _fixed_fit(values, size):
    """theta0, theta1, 0, 0 of each fixed partition by least squares around its first value and middle index."""
    n = values.numel()
    out = []
    for part in (values[:n // size * size].view(-1, size), values[n // size * size:].view(1, -1)):
        if part.numel() == 0:
            continue
        m = part.shape[1]
        x = torch.arange(m, device="cuda", dtype=torch.float64) - (m - 1) / 2
        y = (part - part[:, :1]).to(torch.float64)
        t1 = (y * x).sum(1) / max(float((x * x).sum()), 1.0)
        t0 = part[:, 0].to(torch.float64) + y.mean(1) - t1 * ((m - 1) / 2)
        out.append(torch.stack([t0, t1, torch.zeros_like(t0), torch.zeros_like(t0)], 1).reshape(-1))
    return torch.cat(out)


def exact(case, seed):
    """Decoded values are the column itself; fitted lines are least squares in 64 bits."""
    kind = case["kind"]
    if kind == "batch":
        buffers, parts = _batch_outputs(case)
        for p, v in zip(parts, _batch_columns(case, seed)):
            p.copy_(v)
        return [buffers[False], buffers[True]]
    values = _signed(_values(case, seed))
    if kind == "decode":
        return values
    if kind == "blob":
        return [None, values]
    if kind == "lookup":
        return values[_positions(case, seed).to(torch.int64)]
    if case["part"] != "fixed":
        return None
    n, size = case["n"], case["size"]
    start = torch.arange(0, n, size, device="cuda", dtype=torch.int32)
    return [start, (start.to(torch.int64) + size).clamp_(max=n).to(torch.int32), None,
            _fixed_fit(values.to(torch.int64), size), None, None, None, None]
