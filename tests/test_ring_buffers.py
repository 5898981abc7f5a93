"""Submissions of different kinds and sizes in turn on one ring: buffers that
one kind grows are those that another's captured steps use.  Exact: sets of
whole numbers."""
import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu

RUNS = np.array([0, 40, 9000, 20000], np.uint32)   # partitions: 1, 140 and 172 blocks


@pytest.fixture(scope="module")
def table():
    g = tm.Generator(seed=0xB0F)
    w, ko, k = tm.canonicalize(*g.filters(22000))
    w, ko = np.ascontiguousarray(w[:20000]), ko[:20001]
    k = k[:int(ko[-1])]
    return (w, ko, k), tm.fib_from_runs(w, ko, k, RUNS)[0]


def queries(n, first):
    return tm.Generator(seed=0xB0F).queries(n, 22000, first=first)[0]


def ordered(o, v):
    qid = np.repeat(np.arange(len(o) - 1, dtype=np.uint64), np.diff(o.astype(np.int64)))
    return np.sort((qid << np.uint64(32)) | v)


def check(ring, exp, what):
    o, v = ring.results()
    eo, ev = exp
    assert np.array_equal(o, eo), what
    assert np.array_equal(ordered(o, v), ordered(eo, ev)), what


def unit_lists(tab, q, part, off, mode):
    """The oracle over each unit's partition."""
    w, ko, k = tab
    offs, vals = [np.zeros(1, np.uint64)], []
    for u, p in enumerate(part):
        f0, f1 = int(RUNS[p]), int(RUNS[p + 1])
        eo, ev = orc.match(w[f0:f1], ko[f0:f1 + 1] - ko[f0], k[int(ko[f0]):int(ko[f1])], q[off[u]:off[u + 1]], mode=mode)
        offs.append(eo[1:] + offs[-1][-1])
        vals.append(ev + np.uint32(f0) if mode == 2 else ev)
    return np.concatenate(offs), np.concatenate(vals)


LISTS = [(tm.MODE_HITS, 2), (tm.MODE_KEYS_ALL, 1)]


@pytest.mark.parametrize("mode,om", LISTS)
def test_replays_between_units(gpu, table, mode, om):
    """A captured step is replayed after units have grown the counts that
    both keep by segment and query, twice."""
    tab, fib = table
    ring = tm.Ring(fib, 6000, mode=mode, use_graph=1)
    part = np.array([2, 1, 0, 1], np.uint32)
    q0 = queries(60, 1)
    small = orc.match(*tab, q0, mode=om)
    for n in (1500, 6000):
        for _ in range(2):
            ring.submit(q0)
            ring.wait()
            check(ring, small, f"mode {mode}: 60 queries before {n} in units")
        off = np.array([0, n // 2, n - 10, n - 5, n], np.uint32)
        q = queries(n, n)
        print(f"mode {mode}: {n} queries in units", flush=True)
        ring.submit_units(q, part, off)
        ring.wait()
        check(ring, unit_lists(tab, q, part, off, om), f"mode {mode}: {n} queries in units")
        for turn in range(3):
            ring.submit(q0)
            ring.wait()
            check(ring, small, f"mode {mode}: 60 queries after {n} in units, turn {turn}")
