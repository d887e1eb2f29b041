"""The merge pass of the GPU split/merge partitioner (k_sm_grow, k_sm_more, k_sm_walk and
the chain kernels of g-leco_amd/csrc/glc_splitmerge.hip) as a model: every
partition's group is grown at once for a bounded number of steps, the walk from
partition 0 completes the groups left open where it reaches them, and pointer
doubling in chunks marks the groups of that walk.  Its claim: for ANY merge
decision that depends only on the group's first partition and the candidate
(compression/CpuPartitioner.cuh:207-236) the marked groups are those of the plain
sequential walk, for every bound and chunk length."""
import random

import pytest


def sequential_walk(P, merge):
    starts, g = [0], 0
    for i in range(1, P):
        if not merge(g, i):
            starts.append(i)
            g = i
    return starts


def grow(P, merge, bound):
    """k_sm_grow: first partition after each group, and whether it is open."""
    gend, left = [], []
    for e in range(P):
        j, is_open, steps = e + 1, True, 0
        while is_open and j < P and steps < bound:
            steps += 1
            is_open = merge(e, j)
            j += is_open
        gend.append(j)
        left.append(is_open and j < P)
    return gend, left


def finish(P, merge, gend, left, cand, win):
    """k_sm_walk and k_sm_more in turn: open groups grown on by up to `cand` candidates at a time."""
    e, first = 0, True
    while True:
        if not first:  # k_sm_more, then the first part of k_sm_walk
            assert e < P and j < P
            pays = [merge(e, i) for i in range(j, min(j + min(max(j - e, 1), cand), P))]
            end = pays.index(False) if False in pays else len(pays)
            if end == len(pays) and j + end < P:
                j += end
                continue
            gend[e], left[e] = j + end, False
            e = j + end
        first, wb = False, e - win
        while e < P:
            if e >= wb + win:
                wb = e
                nxt = [-gend[wb + q] if left[wb + q] else gend[wb + q] for q in range(win) if wb + q < P]
            if nxt[e - wb] < 0:
                j = -nxt[e - wb]
                break
            e = nxt[e - wb]
        else:
            return


def chunk_double(s, cnt):
    t = [s[x] if x < cnt else x for x in s]
    inside = any(x < cnt for x in t)
    s[:] = t
    return inside


def chain(P, gend, chunk):
    """k_sm_chain_exit, _walk and _mark (one chunk: k_sm_chain_small)."""
    C = (P + chunk - 1) // chunk
    exits = []
    for b in range(C):
        base, cnt = b * chunk, min(chunk, P - b * chunk)
        s = [gend[base + i] - base for i in range(cnt)]
        more = any(x < cnt for x in s)
        while more:
            more = chunk_double(s, cnt)
        exits += [base + x for x in s]
    entry, e = [-1] * C, 0
    while e < P:
        entry[e // chunk] = e
        e = exits[e]
    mark = []
    for b in range(C):
        base, cnt = b * chunk, min(chunk, P - b * chunk)
        s = [gend[base + i] - base for i in range(cnt)]
        m = [entry[b] >= 0 and base + i == entry[b] for i in range(cnt)]
        more = entry[b] >= 0 and any(x < cnt for x in s)
        while more:
            for i in [i for i in range(cnt) if m[i] and s[i] < cnt]:
                m[s[i]] = True
            more = chunk_double(s, cnt)
        mark += m
    return [i for i in range(P) if mark[i]]


def decision_rule(seed, style):
    memo, rng = {}, random.Random(seed)

    def merge(g, i):
        if (g, i) not in memo:
            p = {0: 0.3, 1: 0.9, 2: 0.995 if (g // 50) % 2 else 0.05, 3: 1.0}[style]
            memo[(g, i)] = rng.random() < p
        return memo[(g, i)]

    return merge


@pytest.mark.parametrize("style", [0, 1, 2, 3])
def test_groups_equal_the_sequential_walk(style):
    for seed in range(25):
        P = random.Random(seed * 11 + style).randint(1, 200)
        merge = decision_rule(seed * 5 + style, style)
        want = sequential_walk(P, merge)
        for bound, cand, win in ((1, 16, 64), (3, 4, 1), (10, 2, 7), (1 << 30, 16, 64)):
            gend, left = grow(P, merge, bound)
            assert all(e < j <= P for e, j in enumerate(gend))  # the chain ends on a provisional list too
            if any(left):
                chain(P, gend, 8)
                finish(P, merge, gend, left, cand, win)
            for chunk in (1, 8, 1 << 20):
                got = chain(P, gend, chunk)
                assert got == want, (seed, style, bound, chunk)
                assert [gend[a] for a in got] == want[1:] + [P]
                assert not any(left[a] for a in got)
