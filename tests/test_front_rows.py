"""The pass before the match (partition counts, rows started from filters with
long key lists) where it can go wrong: query counts around its teams (8, 16),
groups (64) and workgroups, key counts around its four-word loads, filters
that hold every key before and among others, more partitions than are counted
at a time.  Exact: sets of whole numbers."""
import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


def table(n, n_keys, n_full, n_long, seed):
    """n filters of 1-4 keys, but n_full that hold every key and n_long that
    hold a third of them; the empty and the full filter among the latter."""
    rng = np.random.default_rng(seed)
    w, _, _ = tm.Generator(seed=0xF00 + seed).filters(n)
    w[0], w[1] = 0, 0xFFFFFFFF
    w = np.unique(w, axis=0)
    cnt = rng.integers(1, 5, len(w))
    which = 1 + rng.choice(len(w) - 2, n_full + n_long, replace=False)
    cnt[which[:n_full]] = n_keys
    cnt[which[n_full:]] = n_keys // 3
    if n_long:
        cnt[0] = cnt[-1] = n_keys // 3
    ko = np.zeros(len(w) + 1, np.uint64)
    np.cumsum(cnt, out=ko[1:])
    k = np.concatenate([rng.choice(n_keys, c, replace=False) for c in cnt]).astype(np.uint32) * 3 + 2
    return tm.canonicalize(w, ko, k)


def queries(n, seed):
    q, _ = tm.Generator(seed=0xF00 + seed).queries(n, 900, first=5)
    q[n // 2] = 0xFFFFFFFF
    if n > 2:
        q[n // 3] = 0
    return q


def lists(rows, dictionary):
    bits = np.unpackbits(rows.view(np.uint8), axis=1, bitorder="little")
    return bits.sum(1), dictionary[np.nonzero(bits)[1]]


@pytest.mark.parametrize("n_keys,n_full,n_long", [(96, 70, 30), (127, 1, 0), (2048, 9, 60), (2050, 0, 300),
                                                  (6400, 3, 90), (200, 0, 1100)])
def test_rows_vs_oracle(gpu, n_keys, n_full, n_long):
    cw, ko, k = table(2000, n_keys, n_full, n_long, n_keys)
    fib, *_ = tm.build_fib(cw, ko, k, 500)
    for nq in (1, 7, 8, 9, 17, 64, 65, 4097, 5000):
        q = queries(nq, nq)
        print(f"keys {n_keys} full {n_full} long {n_long} queries {nq}", flush=True)
        eo, ev = orc.match(cw, ko, k, q, mode=0)
        for cfg in ({}, {"full_exit": 2}):
            o, v, _ = tm.match(fib, q, mode=tm.MODE_KEYS_UNIQUE, **cfg)
            assert np.array_equal(o, eo) and np.array_equal(v, ev), (nq, cfg)
        r = tm.Ring(fib, nq, mode=tm.MODE_KEYS_UNIQUE)
        r.submit(q)
        r.wait()
        cnt, keys = lists(r.key_bitmaps(), np.unique(k))
        assert np.array_equal(cnt, np.diff(eo.astype(np.int64))) and np.array_equal(keys, ev), nq


def test_large_steps_equal_small_ones(gpu):
    """More than a wave's 64 queries for each wave of a workgroup, and more
    than the queries that its list takes at a time."""
    cw, ko, k = table(1500, 96, 4, 60, 3)
    fib, *_ = tm.build_fib(cw, ko, k, 500)
    q = queries(1021, 1)
    eo, ev = orc.match(cw, ko, k, q, mode=0)
    for times in (300, 1100):
        print(f"{times} x {len(q)} queries", flush=True)
        o, v, _ = tm.match(fib, np.tile(q, (times, 1)), mode=tm.MODE_KEYS_UNIQUE)
        assert np.array_equal(np.diff(o), np.tile(np.diff(eo), times)) and np.array_equal(v, np.tile(ev, times))


@pytest.mark.parametrize("nq", [1, 65, 5000])
def test_counts_of_many_partitions(gpu, nq):
    """5000 partitions, counted 2048 at a time."""
    cw, ko, k = table(6000, 96, 0, 20, 4)
    off = np.unique(np.linspace(0, len(cw), 5001).astype(np.uint32))
    fib, _ = tm.fib_from_runs(cw, ko, k, off)
    q = queries(nq, 2)
    r = tm.Ring(fib, nq, mode=tm.MODE_KEYS_UNIQUE)
    r.submit(q)
    r.wait()
    m = np.stack([np.bitwise_and.reduce(cw[a:b], axis=0) for a, b in zip(off[:-1], off[1:])])
    exp = np.array([((x & ~q) == 0).all(axis=1).sum() for x in m])
    assert np.array_equal(r.lookup_counts()[:len(exp)], exp)
    eo, ev = orc.match(cw, ko, k, q, mode=0)
    o, v = r.results()
    assert np.array_equal(o, eo) and np.array_equal(v, ev)
