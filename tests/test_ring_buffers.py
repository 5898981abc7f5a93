"""Submissions of different kinds and sizes in turn on one ring: buffers that
one kind grows are those that another's captured steps use.  Exact: sets of
whole numbers."""
import ctypes as C

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


def free_memory():
    """Bytes of device memory left (the HIP runtime that the library uses)."""
    free, total = C.c_size_t(), C.c_size_t()
    assert tm.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


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


@pytest.mark.parametrize("mode,om", LISTS)
def test_replayed_hit_list_outgrown_after_units(gpu, table, mode, om):
    """A captured step with a hit list (work items logged) has more hits than
    the list holds, with units in between, which keep none: it is run again."""
    tab, fib = table
    few, fit, many = np.zeros((64, 6), np.uint32), np.zeros((64, 6), np.uint32), queries(64, 3)
    few[:4] = queries(4, 7)
    fit[:2] = 0xFFFFFFFF
    many[:5] = 0xFFFFFFFF
    exp_few, exp_many = orc.match(*tab, few, mode=om), orc.match(*tab, many, mode=om)
    ring = tm.Ring(fib, 64, mode=mode, use_graph=1, log_units=1, hit_capacity=41000)
    part, off = np.array([1], np.uint32), np.array([0, 4], np.uint32)

    def units():
        ring.submit_units(few[:4], part, off)
        assert ring.wait().overflow == 0
        check(ring, unit_lists(tab, few[:4], part, off, om), f"mode {mode}: units")

    units()                 # their counts do not grow again
    ring.submit(fit)        # 40000 hits: the ring's values have room for those of a full hit list
    ring.wait()
    check(ring, orc.match(*tab, fit, mode=om), f"mode {mode}: as many hits as the list holds")
    for _ in range(2):
        ring.submit(few)
        assert ring.wait().overflow == 0
        check(ring, exp_few, f"mode {mode}: few hits")
    units()
    ring.submit(many)
    st = ring.wait()
    assert st.overflow == 1 and st.hit_capacity >= st.n_hits >= 100000
    check(ring, exp_many, f"mode {mode}: many hits")


def test_hits_take_no_list_memory(gpu, table):
    """HITS values are written in place: 40M of them take their own memory
    (4 bytes and a quarter more), none for a hit list (8 bytes)."""
    tab, fib = table
    n = 2000
    q = np.full((n, 6), 0xFFFFFFFF, np.uint32)
    ring = tm.Ring(fib, n, mode=tm.MODE_HITS, hit_capacity=1000)
    before = free_memory()
    ring.submit(q)
    st = ring.wait()
    used = before - free_memory()
    print(f"{st.n_hits} hits, {used / 1e6:.0f} MB", flush=True)
    assert st.n_hits == st.n_results == n * 20000
    assert st.overflow == 1 and st.hit_capacity >= st.n_hits
    assert used < 5 * st.n_hits + (64 << 20)
    ring.submit_resident(n)
    assert ring.wait().overflow == 0
    o, v = ring.results()
    assert np.array_equal(np.sort(v[:20000]), np.arange(20000)) and int(o[1]) == 20000


def test_units_cut_into_whole_tiles(gpu, table):
    """Segments of fewer blocks than a tile (32) make no items without any."""
    tab, fib = table
    part, off = np.array([0, 1, 2], np.uint32), np.array([0, 3, 73, 100], np.uint32)
    q = queries(100, 5)
    for seg in (1, 4, 31, 33, 0):
        ring = tm.Ring(fib, 100, mode=tm.MODE_KEYS_UNIQUE, chunk_blocks=seg)
        ring.submit_units(q, part, off)
        st = ring.wait()
        tiles = 1 + 2 * 5 + 6      # of 1, 140 and 172 blocks, for 3, 70 (64 and 6) and 27 queries
        print(f"segment {seg}: {st.n_items} items", flush=True)
        assert st.n_items <= tiles, seg
        check(ring, unit_lists(tab, q, part, off, 0), f"segment {seg}")


@pytest.mark.parametrize("mode,om", LISTS)
def test_unit_counts_are_bounded(gpu, mode, om):
    """Units in the list modes: counts by segment and query take 256 MB at
    most, however many queries and however small the segments."""
    g = tm.Generator(seed=0xB0F)
    w, ko, k = tm.canonicalize(*g.filters(240000))
    n, nq = 200000, 800000     # 98 segments of 32 blocks x 800k queries: 314 MB
    w, ko = np.ascontiguousarray(w[:n]), ko[:n + 1]
    k = k[:int(ko[-1])]
    assert w[0].any()          # no empty filter: the empty query matches nothing
    fib, _ = tm.fib_from_runs(w, ko, k, np.array([0, n], np.uint32))
    q = np.zeros((nq, 6), np.uint32)
    at = np.arange(40) * 20011
    q[at] = g.queries(40, 240000)[0]
    ring = tm.Ring(fib, nq, mode=mode, chunk_blocks=32, hit_capacity=1000)
    before = free_memory()
    ring.submit_units(q, np.zeros(1, np.uint32), np.array([0, nq], np.uint32))
    st = ring.wait()
    used = before - free_memory()
    print(f"mode {mode}: {st.n_hits} hits, {used / 1e6:.0f} MB", flush=True)
    eo, ev = orc.match(w, ko, k, q[at], mode=om)
    o, v = ring.results()
    assert np.array_equal(np.diff(o.astype(np.int64))[at], np.diff(eo.astype(np.int64)))
    assert int(o[-1]) == len(ev) and np.array_equal(np.sort(v), np.sort(ev))
    assert used <= (256 << 20) + (32 << 20)


def test_few_configured_segments(gpu):
    """Few segments, configured: items of fewer queries, so that the GPU is
    not left idle (and the counts by segment and query agree with the shape
    that the kernel takes)."""
    g = tm.Generator(seed=0xB0F)
    tab = tm.canonicalize(*g.filters(100000))
    fib, *_ = tm.build_fib(*tab, 30000)
    nq = 150000
    q = np.zeros((nq, 6), np.uint32)
    at = np.arange(60) * 2477
    q[at] = g.queries(60, 100000)[0]
    for mode, om in LISTS:
        eo, ev = orc.match(*tab, q[at], mode=om)
        for seg in (64, 1000, 4096):
            ring = tm.Ring(fib, nq, mode=mode, chunk_blocks=seg)
            ring.submit(q)
            st = ring.wait()
            o, v = ring.results()
            print(f"mode {mode} segment {seg}: {st.n_items} items", flush=True)
            assert np.array_equal(np.diff(o.astype(np.int64))[at], np.diff(eo.astype(np.int64)))
            got = [np.sort(v[int(o[i]):int(o[i + 1])]) for i in at]
            want = [np.sort(ev[int(eo[i]):int(eo[i + 1])]) for i in range(60)]
            assert all(np.array_equal(x, y) for x, y in zip(got, want))
            assert st.n_items >= 400


def test_groups_per_cu_holds(gpu):
    """groups_per_cu bounds the workgroups that a step is cut for: a small
    step, one item each, makes about half as many items with one per CU as
    with two."""
    g = tm.Generator(seed=0xB0F)
    tab = tm.canonicalize(*g.filters(800000))
    fib, *_ = tm.build_fib(*tab, 60000)
    q = queries(500, 3)
    items, res = [], []
    for groups in (0, 2, 1):
        ring = tm.Ring(fib, 500, mode=tm.MODE_HITS, groups_per_cu=groups)
        ring.submit(q)
        items.append(ring.wait().n_items)
        res.append(ring.results())
        assert np.array_equal(res[0][0], res[-1][0])
        assert np.array_equal(ordered(*res[0]), ordered(*res[-1]))
    print(f"items {items}", flush=True)
    assert items[0] == items[1] and items[2] < 0.7 * items[1]


ALL_MODES = LISTS + [(tm.MODE_KEYS_UNIQUE, 0)]


@pytest.mark.parametrize("mode,om", ALL_MODES)
def test_units_of_few_blocks_are_spread(gpu, table, mode, om):
    """1000 queries on one small partition: more than a few items."""
    tab, fib = table
    q = queries(1063, 9)
    for part, n in ((0, 1000), (1, 1063), (0, 65), (0, 64)):
        ring = tm.Ring(fib, n, mode=mode)
        p, off = np.array([part], np.uint32), np.array([0, n], np.uint32)
        ring.submit_units(q[:n], p, off)
        st = ring.wait()
        print(f"mode {mode} partition {part}: {n} queries, {st.n_items} items", flush=True)
        check(ring, unit_lists(tab, q[:n], p, off, om), f"mode {mode} partition {part} queries {n}")
        assert st.n_items >= n // 64


@pytest.mark.parametrize("mode,om", ALL_MODES)
def test_steps_on_few_blocks_are_spread(gpu, mode, om):
    """1000 queries on a table of 1000 filters: more than a few items."""
    g = tm.Generator(seed=0xB0F)
    tab = tm.canonicalize(*g.filters(1000))
    fib, _ = tm.fib_from_runs(*tab, np.array([0, len(tab[0])], np.uint32))   # 15 blocks
    for n in (1000, 1025, 65, 64, 3):
        q = queries(n, 31)
        ring = tm.Ring(fib, n, mode=mode, full_exit=2)
        ring.submit(q)
        st = ring.wait()
        print(f"mode {mode}: {n} queries, {st.n_items} items", flush=True)
        check(ring, orc.match(*tab, q, mode=om), f"mode {mode} queries {n}")
        assert st.n_items >= n // 64


def test_results_after_a_refused_submission(gpu):
    """A submission that the table's growth makes impossible (more keys than
    rows can hold) leaves the last one's lists: those of its first queries."""
    w, _, _ = tm.Generator(seed=0xB0F).filters(48000)
    w = np.unique(w, axis=0)[:35100]
    small = tm.canonicalize(w, np.arange(len(w) + 1, dtype=np.uint64), (np.arange(len(w)) % 3000).astype(np.uint32))
    large = tm.canonicalize(w, np.arange(0, 2 * len(w) + 1, 2, dtype=np.uint64), np.arange(2 * len(w), dtype=np.uint32))
    off, mask = np.array([0, len(w)], np.uint32), np.zeros((1, 6), np.uint32)
    fib = tm.Fib(small[0], off, mask, small[1], small[2])
    q = queries(5000, 77)
    exp = orc.match(*small, q, mode=0)
    ring = tm.Ring(fib, 5000, mode=tm.MODE_KEYS_UNIQUE)
    ring.submit(q[-5:])      # lists in host memory, then more than it takes
    ring.wait()
    ring.submit(q)
    ring.wait()
    check(ring, exp, "before the upload")
    fib.upload(large[0], off, mask, large[1], large[2])
    with pytest.raises(tm.TagMatchError):
        ring.submit(q[:20])
    o, v = ring.results()
    assert np.array_equal(o, exp[0][:21]) and np.array_equal(v, exp[1][:int(exp[0][20])])
