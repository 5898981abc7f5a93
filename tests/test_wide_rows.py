"""Key rows of more than 64 words (2048 keys), whose items hold fewer queries
the wider they are: 96 at 4096 keys, 47 at 8200, 15 at 24600, 6 at 65000.
Units around those sizes with one and several segments, with and without long
key lists, and steps that start from empty rows.  Exact: sets of whole
numbers."""
import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


def table(n, n_keys, long_lists, seed=3):
    """n canonical filters with 1-4 keys, but long_lists of them with 33-300;
    every key occurs."""
    rng = np.random.default_rng(seed)
    w, _, _ = tm.Generator(seed=0x31DE + seed).filters(n + n // 4 + 100)
    w = np.unique(w, axis=0)[:n]
    cnt = rng.integers(1, 5, n)
    if long_lists:
        at = rng.choice(n, long_lists, replace=False)
        cnt[at] = rng.integers(33, 301, long_lists)
    ko = np.zeros(n + 1, np.uint64)
    np.cumsum(cnt, out=ko[1:])
    k = np.concatenate([rng.choice(n_keys, c, replace=False) for c in cnt]).astype(np.uint32)
    first = ko[:-1].astype(np.int64)
    for i in range(0, n_keys, n):      # the first key of the filters: all of them in turn
        some = np.arange(i, min(i + n, n_keys))
        k[first[:len(some)] + (i // n) % cnt[:len(some)]] = some
    return tm.canonicalize(w, ko, k)


def queries(n, n_filters, seed=3):
    q = tm.Generator(seed=0x31DE + seed).queries(n, n_filters, first=99)[0]
    q[n // 2] = 0xFFFFFFFF
    return q


@pytest.mark.parametrize("n_keys,long_lists", [(4096, 30), (8200, 30), (8200, 0), (24600, 30), (24600, 0), (65000, 9)])
def test_units_of_wide_rows(gpu, n_keys, long_lists):
    cw, ko, k = table(9000, n_keys, long_lists)
    off = np.array([0, 100, 2500, len(cw)], np.uint32)   # 2, 38 and 102 blocks
    fib, _ = tm.fib_from_runs(cw, ko, k, off)
    most = 12288 // ((len(np.unique(k)) + 31) // 32)      # queries of an item
    sizes = [most - 1, most, most + 1, 1, 3 * most + 1, 200]
    part = np.array([0, 1, 2, 2, 1, 2], np.uint32)
    uo = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    q = queries(int(uo[-1]), len(cw))
    for seg in (0, 32):
        ring = tm.Ring(fib, len(q), mode=tm.MODE_KEYS_UNIQUE, chunk_blocks=seg)
        for turn in range(2):
            print(f"keys {n_keys} lists {long_lists} segment {seg} turn {turn}", flush=True)
            ring.submit_units(q, part, uo)
            ring.wait()
            o, v = ring.results()
            for u, p in enumerate(part):
                f0, f1, a, b = int(off[p]), int(off[p + 1]), int(uo[u]), int(uo[u + 1])
                eo, ev = orc.match(cw[f0:f1], ko[f0:f1 + 1] - ko[f0], k[int(ko[f0]):int(ko[f1])], q[a:b], mode=0)
                assert np.array_equal(o[a:b + 1] - o[a], eo), (u, seg)
                assert np.array_equal(v[int(o[a]):int(o[b])], ev), (u, seg)


@pytest.mark.parametrize("n_keys", [4096, 8200, 16384, 24600])
def test_steps_from_empty_rows(gpu, n_keys):
    """No filter with a long list: rows start empty."""
    cw, ko, k = table(9000, n_keys, 0)
    fib, *_ = tm.build_fib(cw, ko, k, 1500)
    for nq in (1, 23, 48, 97, 1300):
        print(f"keys {n_keys} queries {nq}", flush=True)
        q = queries(nq, len(cw))
        eo, ev = orc.match(cw, ko, k, q, mode=0)
        for fe in (0, 2):
            o, v, _ = tm.match(fib, q, full_exit=fe)
            assert np.array_equal(o, eo) and np.array_equal(v, ev), (nq, fe)


def test_steps_from_empty_rows_by_size(gpu):
    """The sizes between which steps from empty rows change kernels (8192
    keys, about 6300 blocks: 3.8k, 11k and 12k queries), against the step with
    the exit, and the oracle on a sample."""
    cw, ko, k = table(400_000, 8192, 0)
    fib, *_ = tm.build_fib(cw, ko, k, 30_000)
    q = queries(12500, len(cw))
    at = np.linspace(0, 3699, 60).astype(np.int64)
    eo, ev = orc.match(cw, ko, k, q[at], mode=0)
    for nq in (3700, 5000, 11800, 12500):
        print(f"queries {nq}", flush=True)
        o, v, _ = tm.match(fib, q[:nq], full_exit=2)
        o1, v1, _ = tm.match(fib, q[:nq])
        assert np.array_equal(o, o1) and np.array_equal(v, v1)
        got = np.concatenate([v[int(o[i]):int(o[i + 1])] for i in at])
        assert np.array_equal(np.diff(o.astype(np.int64))[at], np.diff(eo.astype(np.int64))) and np.array_equal(got, ev)


def test_unit_time_does_not_jump_with_the_dictionary(gpu):
    """4096 keys against 2048, the same filters, lists and units: rows twice
    the width, at most five times the match time."""
    ms = []
    for n_keys in (2048, 4096):
        cw, ko, k = table(200_000, n_keys, 300)
        fib, _ = tm.fib_from_runs(cw, ko, k, np.array([0, 60_000, len(cw)], np.uint32))
        q = queries(4000, len(cw))
        ring = tm.Ring(fib, len(q), mode=tm.MODE_KEYS_UNIQUE)
        part, uo = np.array([0, 1], np.uint32), np.array([0, 1500, 4000], np.uint32)
        t = []
        for _ in range(6):
            ring.submit_units(q, part, uo)
            t.append(ring.wait().match_ms)
        ms.append(float(np.median(t)))
    print(f"match ms {ms}", flush=True)
    assert ms[1] < 5 * ms[0]
