"""Steps whose queries are taken, and whose lists are delivered, by their own
kernels: at the sizes where the copies take over (4096 queries, 8192 values),
replayed with changing and with resident queries, and after a refused
submission.  Exact: sets of whole numbers."""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def table():
    g = tm.Generator(seed=0x57E9)
    return tm.canonicalize(*g.filters(3000))


def queries(n, first):
    return tm.Generator(seed=0x57E9).queries(n, 3000, first=first)[0]


def ordered(o, v):
    qid = np.repeat(np.arange(len(o) - 1, dtype=np.uint64), np.diff(o.astype(np.int64)))
    return np.sort((qid << np.uint64(32)) | v)


MODES = [(tm.MODE_KEYS_UNIQUE, 0), (tm.MODE_HITS, 2)]


@pytest.mark.parametrize("mode,om", MODES)
@pytest.mark.parametrize("sched", [tm.SCHED_PERSISTENT, tm.SCHED_PLAIN])
def test_lists_where_copies_take_over(gpu, table, mode, om, sched):
    cw, ko, k = table
    fib, *_ = tm.build_fib(cw, ko, k, 700)
    q = queries(5000, 11)
    eo, ev = orc.match(cw, ko, k, q, mode=om)
    full = int(np.searchsorted(eo, 8193)) - 1     # the most queries of at most 8192 values
    ring = tm.Ring(fib, 5000, mode=mode, schedule=sched)
    for nq in (1, full, full + 1, 4095, 4096, 4097, 5000, 2):
        print(f"mode {mode} schedule {sched} queries {nq} values {int(eo[nq])}", flush=True)
        ring.submit(q[:nq])
        assert ring.wait().n_results == int(eo[nq])
        o, v = ring.results()
        assert np.array_equal(o, eo[:nq + 1])
        assert np.array_equal(ordered(o, v), ordered(eo[:nq + 1], ev[:int(eo[nq])]))


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("mode,om", MODES)
def test_submitted_and_resident_queries_in_turn(gpu, table, mode, om, graph):
    """A replay takes the queries of its own submission, and leaves those that
    another program put into the ring's buffer alone."""
    cw, ko, k = table
    fib, *_ = tm.build_fib(cw, ko, k, 700)
    ring = tm.Ring(fib, 128, mode=mode, use_graph=graph)
    buf = C.c_void_p()
    lib = tm.load()
    tm.check(lib.tm_ring_query_buffer(ring.h, C.byref(buf)), "tm_ring_query_buffer")
    for turn in range(4):
        for n, resident in ((128, False), (128, True), (100, False), (64, True)):
            q = queries(n, 1000 * turn + n + resident)
            if resident:
                w = np.zeros((n, 8), np.uint32)
                w[:, :6] = q
                tm.check(lib.tm_dev_upload(buf, w.ctypes.data_as(C.c_void_p), w.nbytes), "tm_dev_upload")
                ring.submit_resident(n)
            else:
                ring.submit(q)
            ring.wait()
            o, v = ring.results()
            eo, ev = orc.match(cw, ko, k, q, mode=om)
            assert np.array_equal(o, eo), (turn, n, resident)
            assert np.array_equal(ordered(o, v), ordered(eo, ev)), (turn, n, resident)


def test_queries_of_a_refused_submission_are_resident(gpu, table):
    cw, ko, k = table
    fib, *_ = tm.build_fib(cw, ko, k, 700)
    kw = (int(fib.stats()["n_distinct_keys"]) + 31) // 32
    q = queries(50, 5)
    ring = tm.Ring(fib, 64, mode=tm.MODE_KEY_BITMAP)
    ring.set_host_rows(tm.PinnedRows(10 * kw))
    with pytest.raises(tm.TagMatchError):
        ring.submit(q)
    ring.set_host_rows(tm.PinnedRows(64 * kw))
    ring.submit_resident(50)
    ring.wait()
    rows = ring.key_bitmaps()
    eo, ev = orc.match(cw, ko, k, q, mode=0)
    bits = np.unpackbits(rows.view(np.uint8), axis=1, bitorder="little")
    assert np.array_equal(bits.sum(1), np.diff(eo.astype(np.int64)))
    assert np.array_equal(np.unique(k)[np.nonzero(bits)[1]], ev)
