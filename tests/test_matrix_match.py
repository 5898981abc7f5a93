"""The matrix-core match against the oracle at the sizes where it can go
wrong: query counts around its tiles (32), pairs (64) and work items (192,
1536, 2048), rows in local memory and in HBM (2048 and 2080 keys), partly
filled blocks, the empty and the full filter and query, and more filters with
long key lists than the rich-filter pass takes.  Exact: sets of whole
numbers."""
import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


def table(n, n_keys, long_lists, seed):
    """n canonical filters, every other one with 1-4 keys, `long_lists` of
    them with 33-130; the empty and the full filter among them."""
    rng = np.random.default_rng(seed)
    g = tm.Generator(seed=0x5EED + seed)
    w, _, _ = g.filters(n)
    w[0], w[1] = 0, 0xFFFFFFFF
    w = np.unique(w, axis=0)
    cnt = rng.integers(1, 5, len(w))
    cnt[rng.choice(len(w), min(long_lists, len(w)), replace=False)] = rng.integers(33, 131, min(long_lists, len(w)))
    ko = np.zeros(len(w) + 1, np.uint64)
    cnt = np.minimum(cnt, n_keys)
    np.cumsum(cnt, out=ko[1:])
    k = np.concatenate([rng.choice(n_keys, c, replace=False) for c in cnt]).astype(np.uint32) * 5 + 1
    return tm.canonicalize(w, ko, k)


def queries(n, seed):
    q, _ = tm.Generator(seed=0x5EED + seed).queries(n, 4000, first=77)
    q[n // 2] = 0xFFFFFFFF
    if n > 2:
        q[n // 3] = 0
    return q


def same(got, exp, what, ordered):
    (go, gv), (eo, ev) = got, exp
    assert np.array_equal(go, eo), what
    if not ordered:
        qid = np.repeat(np.arange(len(go) - 1, dtype=np.uint64), np.diff(go.astype(np.int64)))
        gv = (np.sort((qid << np.uint64(32)) | gv) & np.uint64(0xFFFFFFFF)).astype(np.uint32)
        ev = (np.sort((qid << np.uint64(32)) | ev) & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    assert np.array_equal(gv, ev), what


MODES = [(tm.MODE_KEYS_UNIQUE, {}, 0), (tm.MODE_KEYS_UNIQUE, {"full_exit": 2}, 0), (tm.MODE_HITS, {}, 2),
         (tm.MODE_KEYS_ALL, {}, 1)]


@pytest.mark.parametrize("n_keys,long_lists", [(2048, 0), (2048, 1100), (2080, 40), (96, 40)])
def test_matrix_match_vs_oracle(gpu, n_keys, long_lists):
    cw, ko, k = table(4000, n_keys, long_lists, n_keys + long_lists)
    fib, *_ = tm.build_fib(cw, ko, k, 700)
    for nq in (1, 31, 32, 33, 64, 65, 191, 193, 1537, 2049):
        q = queries(nq, nq)
        print(f"keys {n_keys} long {long_lists} queries {nq}", flush=True)
        for mode, cfg, om in MODES:
            o, v, st = tm.match(fib, q, mode=mode, **cfg)
            exp = orc.match(cw, ko, k, q, mode=om)
            same((o, v), exp, f"mode {mode} {cfg} nq {nq}", ordered=om == 0)
            if mode == tm.MODE_HITS:
                assert st["n_hits"] == int(exp[0][-1])


@pytest.mark.parametrize("mode,om", [(tm.MODE_KEYS_UNIQUE, 0), (tm.MODE_HITS, 2), (tm.MODE_KEYS_ALL, 1)])
def test_matrix_units_vs_oracle(gpu, mode, om):
    """Explicit units whose query ranges end inside tiles and items."""
    cw, ko, k = table(4000, 2048, 30, 5)
    off = np.array([0, 1, 130, 131, 1500, len(cw)], np.uint32)
    fib, _ = tm.fib_from_runs(cw, ko, k, off)
    sizes = [1, 33, 191, 193, 700, 0, 64]
    part = np.array([0, 1, 2, 3, 4, 3, 4], np.uint32)
    uo = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    q = queries(int(uo[-1]), 9)
    for seg in (0, 64):
        ring = tm.Ring(fib, len(q), mode=mode, chunk_blocks=seg)
        ring.submit_units(q, part, uo)
        ring.wait()
        o, v = ring.results()
        ring.close()
        for u, p in enumerate(part):
            a, b = int(uo[u]), int(uo[u + 1])
            if a == b:
                continue
            f0, f1 = int(off[p]), int(off[p + 1])
            kb = ko[f0:f1 + 1] - ko[f0]
            eo, ev = orc.match(cw[f0:f1], kb, k[int(ko[f0]):int(ko[f1])], q[a:b], mode=om)
            if mode == tm.MODE_HITS:
                ev = ev + np.uint32(f0)
            same((o[a:b + 1] - o[a], v[int(o[a]):int(o[b])]), (eo, ev), f"unit {u} segment {seg}", ordered=om == 0)


def test_rich_marks_of_an_image(gpu, tmp_path):
    """A loaded image keeps the marks of rich filters that are true and drops
    the others: one slot marked as another rich filter still gives its keys."""
    cw, ko, k = table(3000, 2048, 60, 11)
    fib, *_ = tm.build_fib(cw, ko, k, 700)
    q = queries(300, 3)
    exp = orc.match(cw, ko, k, q, mode=0)
    path = tmp_path / "a.fib"
    fib.save(str(path))
    data = bytearray(path.read_bytes())
    pos = 88
    for item in (4, 4):                                  # block words, block info
        pos += 8 + int.from_bytes(data[pos:pos + 8], "little") * item
    n = int.from_bytes(data[pos:pos + 8], "little")
    slots = np.frombuffer(data, np.uint64, n, pos + 8).copy()
    marked = np.flatnonzero(((slots & 0xFFFF) == 0xFFFF) & ((slots >> 48) != 0) & (slots != 0xFFFFFFFFFFFFFFFF))
    assert len(marked) == 60
    s = slots[marked]
    slots[marked] = (s & np.uint64(0xFFFFFFFFFFFF)) | (np.roll(s, 1) >> np.uint64(48) << np.uint64(48))
    data[pos + 8:pos + 8 + n * 8] = slots.tobytes()
    (tmp_path / "b.fib").write_bytes(bytes(data))
    for name in ("a.fib", "b.fib"):
        o, v, _ = tm.match(tm.Fib.from_image(str(tmp_path / name)), q)
        same((o, v), exp, name, ordered=True)
