"""The work that programs built on tagmatch_amd have it do, as timed cases.

Every case goes through the package's public entry points (rings, explicit
units, the no-allocation call, the GPU partitioner, the cost model) on the
tables and queries of the workload generator: 192-bit filters of 1-10 Zipf
tags with 1-4 keys, queries of 10-30 tags, 30% of them supersets of a filter.

listed()             the cases
draw(rng)            one more case of the same ranges
prepare(case, seed)  what a program holds before the call
run(state)           one pass, and everything it computes
work(case)           bytes and operations of one pass that cannot be left out
exact(case, seed)    the 64-bit result where the outputs are computed numbers

Tables do not depend on the seed (a program keeps its table; queries come
and go), so each one is built once per process and kept.  Results come in
sizes that the case fixes: cases whose results are lists of any length take
one stretch of queries in an order made from the seed, the others a stretch
of their own for each seed.
"""
import ctypes as C
from collections import OrderedDict

import numpy as np
import torch

import tagmatch_amd as tm

SEED = 0x7461676D61746302     # the generator seed of the benchmark's table
KEYS = 2048                   # distinct keys of the generated tables (8 trees x 256 interfaces)
KEEP_TABLES = 3               # small tables kept beside those the listed cases use

# n_filters -> largest partition: the 10M and 1M tables of the benchmark's
# configurations and the smoke run's; other tables get about 16 partitions
MAXP = {10_000_000: 256 * 1024, 1_000_000: 64 * 1024, 30_000: 2048}
MAX_PARTS = 4096              # partitions that the partitioning cases leave room for


def _maxp(n_filters):
    return MAXP.get(n_filters, max(1024, n_filters // 16))


def listed():
    return [
        # one message to route as it arrives, small table: its sorted key list on the host
        {"name": "keys_1", "kind": "keys", "filters": 30_000, "queries": 1, "out": "host"},
        # a serving request alone in a slot: a replayed step of 64 queries,
        # key bitmap rows delivered to pinned host memory
        {"name": "serve_64", "kind": "serve", "filters": 1_000_000, "queries": 64},
        # a serving slot nearly full (1024 queries at most, padded replays)
        {"name": "serve_1000", "kind": "serve", "filters": 10_000_000, "queries": 1000},
        # the 1M-filter configuration's 100k queries, key lists kept in HBM
        {"name": "keys_100k", "kind": "keys", "filters": 1_000_000, "queries": 100_000, "out": "device"},
        # rows for queries that another GPU program made, in its own memory,
        # with nothing allocated (a ragged size)
        {"name": "static_9999", "kind": "static", "filters": 10_000_000, "queries": 9_999},
        # the benchmark's headline: 1M resident queries, packed rows to the host
        {"name": "packed_1m", "kind": "packed", "filters": 10_000_000, "queries": 1_000_000},
        # the same queries as sorted key lists left in HBM (8 GB of keys)
        {"name": "keys_1m", "kind": "keys", "filters": 10_000_000, "queries": 1_000_000, "out": "device"},
        # every match enumerated (no full-key-set exit): the matches/s figure;
        # rows to the host
        {"name": "every_match_65k", "kind": "every", "filters": 10_000_000, "queries": 65_536},
        # which filters match, as a cache or an audit asks for them: ids per query
        {"name": "hits_1024", "kind": "hits", "filters": 10_000_000, "queries": 1024},
        # uneven batching: Zipf(1.2) partitions of 1k to 1M filters, eight
        # batches of 1-4096 queries for each
        {"name": "units_uneven", "kind": "units", "filters": 10_000_000, "rounds": 8},
        # balanced partitioning when a table of 1M filters is consolidated
        {"name": "partition_1m", "kind": "partition", "filters": 1_000_000},
        # the cost model's training pass (forward and backward) over a large batch of unit logs
        {"name": "mlp_grad_65k", "kind": "mlp", "rows": 65_536},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["keys", "keys", "serve", "static", "packed", "every", "hits", "keys_all", "units",
                       "partition", "mlp"])
    if kind == "mlp":
        return {"kind": kind, "rows": _log_uniform(rng, 256, 65_536)}
    if kind == "partition":
        return {"kind": kind, "filters": _log_uniform(rng, 30_000, 1_000_000)}
    if kind == "units":
        return {"kind": kind, "filters": _log_uniform(rng, 100_000, 1_000_000), "rounds": rng.randint(1, 8)}
    if kind == "keys":
        case = {"kind": kind, "filters": 0, "queries": _log_uniform(rng, 1, 1_000_000)}
        case["out"] = "host" if case["queries"] <= 512 else "device"
    else:
        top = {"serve": 1024, "static": tm.STATIC_MAX_QUERIES, "packed": 1_000_000, "every": 65_536, "hits": 1024,
               "keys_all": 64}[kind]
        case = {"kind": kind, "filters": 0, "queries": _log_uniform(rng, 16, top)}
    # a handful of queries on a large table nearly always match every key
    nq = case["queries"]
    if (nq >= 512 or kind in ("hits", "keys_all")) and rng.random() < 0.5:
        case["filters"] = 10_000_000
    else:
        case["filters"] = _log_uniform(rng, 30_000, 1_000_000 if nq >= 16 else 300_000)
    return case


# ------------------------------------------------------------------ tables

_tables = OrderedDict()


class _Table:
    """A canonical table of n generated filters; fib() is its partitioned
    form, runs() the same filters cut into Zipf(1.2) partitions."""

    def __init__(self, n):
        tm.init(0)
        self.n = n
        self.gen = tm.Generator(seed=SEED)
        self.words, self.key_off, self.keys = tm.canonicalize(*self.gen.filters(n))
        self._fib = self._runs = None

    def fib(self):
        if self._fib is None:
            self._fib = tm.build_fib(self.words, self.key_off, self.keys, _maxp(self.n))[0]
        return self._fib

    def runs(self):
        if self._runs is None:
            off = tm.zipf_runs(len(self.words), 1000, 1_000_000, s=1.2, seed=3)
            self._runs = (tm.fib_from_runs(self.words, self.key_off, self.keys, off)[0], len(off) - 1)
        return self._runs

    def queries(self, n, seed):
        """n queries of the generator's stream, another stretch for each seed."""
        return self.gen.queries(n, self.n, first=(1 + seed % (1 << 30)) << 21)[0]

    def shuffled(self, n, seed, bounds=None):
        """The stream's first n queries, shuffled by the seed (within each of
        the stretches that `bounds` cuts)."""
        q = self.gen.queries(n, self.n)[0]
        order = np.random.default_rng(seed).random(n)
        if bounds is not None:
            order += np.repeat(np.arange(len(bounds) - 1), np.diff(bounds.astype(np.int64)))
        return q[np.argsort(order)]


def _table(n):
    t = _tables.pop(n, None) or _Table(n)
    _tables[n] = t
    small = [k for k in _tables if k not in MAXP]
    for k in small[:-KEEP_TABLES]:
        del _tables[k]
    return t


# ------------------------------------------------------------------ passes

class _DeviceArray:
    """Device memory of the library, for torch.as_tensor; the tensor keeps
    the array, and so its owner."""

    def __init__(self, owner, ptr, n, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


class _HostArray:
    """uint32 words of a pinned buffer, for np.asarray, which keeps it."""

    def __init__(self, owner, *shape):
        self.owner = owner
        self.__array_interface__ = {"shape": shape, "typestr": "<u4", "data": (owner.ptr, True), "version": 3}


def _device_lists(ring):
    """(offsets, values) of a ring's finished submission where they lie, in HBM."""
    off, vals = C.c_void_p(), C.c_void_p()
    tm.check(tm.load().tm_ring_results_device(ring.h, C.byref(off), C.byref(vals)), "tm_ring_results_device")
    o = torch.as_tensor(_DeviceArray(ring, off.value, ring.nq + 1, "<i8"), device="cuda")
    n = int(o[-1])
    if n == 0:
        return o, torch.empty(0, dtype=torch.int32, device="cuda")
    return o, torch.as_tensor(_DeviceArray(ring, vals.value, n, "<i4"), device="cuda")


def _padded(a, n):
    """A list of at most n entries in an array of n, zeros behind it."""
    out = np.zeros((n,) + a.shape[1:], a.dtype)
    out[:len(a)] = a
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _prepare_mlp(case, seed)
    if kind == "partition":
        tm.init(0)
        n = case["filters"]
        g = tm.Generator(seed=SEED)
        # enough raw filters for n distinct ones (about 8% are duplicates), sorted
        words, _, _ = tm.canonicalize(*g.filters(n + n // 4, first=(1 + seed % (1 << 30)) << 21))
        return {"kind": kind, "words": np.ascontiguousarray(words[:n]), "maxp": _maxp(n)}
    t = _table(case["filters"])
    if kind == "units":
        fib, n_parts = t.runs()
        parts, offs = [], [0]
        for k in range(case["rounds"]):
            up, uo = tm.uneven_units(n_parts, 1, 4096, seed=100 + k)
            parts.append(up)
            offs.extend((offs[-1] + uo[1:].astype(np.int64)).tolist())
        up, uo = np.concatenate(parts).astype(np.uint32), np.array(offs, np.uint32)
        nq = int(uo[-1])
        ring = tm.Ring(fib, nq)
        ring.submit_units(t.shuffled(nq, seed, uo), up, uo)   # the queries stay resident
        ring.wait()
        return {"kind": kind, "ring": ring, "part": up, "off": uo}
    fib, nq = t.fib(), case["queries"]
    fixed = kind in ("static", "serve", "every") or case.get("out") == "host"   # results of a fixed size
    q = t.queries(nq, seed) if fixed else t.shuffled(nq, seed)
    if kind == "static":
        padded = np.zeros((nq, 8), np.uint32)
        padded[:, :6] = q
        kw = (int(fib.stats()["n_distinct_keys"]) + 31) // 32
        return {"kind": kind, "fib": fib, "queries": torch.from_numpy(padded.view(np.int32)).cuda(),
                "rows": torch.empty((nq, kw), dtype=torch.int32, device="cuda")}
    mode = {"keys": tm.MODE_KEYS_UNIQUE, "every": tm.MODE_KEY_BITMAP, "serve": tm.MODE_KEY_BITMAP,
            "packed": tm.MODE_KEY_BITMAP, "hits": tm.MODE_HITS, "keys_all": tm.MODE_KEYS_ALL}[kind]
    kw = (int(fib.stats()["n_distinct_keys"]) + 31) // 32
    state = {"kind": kind, "q": q, "out": case.get("out")}
    ring = tm.Ring(fib, nq, mode=mode, full_exit=2 if kind == "every" else 0, use_graph=int(kind == "serve"))
    if kind in ("serve", "every"):
        state["rows"] = tm.PinnedRows(nq * kw)
        ring.set_host_rows(state["rows"])
    elif kind == "packed":
        state["rows"] = tm.PackedRows(nq, kw)
        ring.set_host_rows_packed(state["rows"])
    # a ring's first submission grows its buffers to the results' size and,
    # for the steps on resident queries, puts the queries there
    ring.submit(q)
    ring.wait()
    state.update(ring=ring, kw=kw)
    return state


def run(state):
    kind = state["kind"]
    if kind == "mlp":
        return state["mlp"].loss_grad(state["x"], state["t"])
    if kind == "partition":
        perm, off, masks = tm.partition(state["words"], state["maxp"])
        return perm, _padded(off, MAX_PARTS + 1), _padded(masks, MAX_PARTS)
    if kind == "static":
        q, rows = state["queries"], state["rows"]
        tm.check(tm.load().tm_match_rows_static(state["fib"].h, C.c_void_p(q.data_ptr()), q.shape[0],
                                                C.c_void_p(rows.data_ptr()),
                                                C.c_void_p(torch.cuda.current_stream().cuda_stream)),
                 "tm_match_rows_static")
        return rows
    ring = state["ring"]
    if kind == "units":
        ring.submit_units(None, state["part"], state["off"])
        ring.wait()
        return _device_lists(ring)
    nq = len(state["q"])
    if kind in ("serve", "every"):
        ring.submit(state["q"])
        ring.wait()
        return np.asarray(_HostArray(state["rows"], nq, state["kw"]))
    if kind == "packed":
        ring.submit_resident(nq)
        n = ring.wait().n_results
        rows = state["rows"]
        return np.asarray(_HostArray(rows.row_of, nq)), np.asarray(_HostArray(rows.rows, n, state["kw"]))
    if kind in ("hits", "keys_all"):
        # a query's list comes in no particular order: sorted per query
        ring.submit(state["q"])
        ring.wait()
        off, vals = _device_lists(ring)
        qid = torch.repeat_interleave(torch.arange(nq, device="cuda"), off.diff(), output_size=vals.numel())
        return off, torch.sort((qid << 32) | (vals.to(torch.int64) & 0xFFFFFFFF)).values
    if state["out"] == "host":
        ring.submit(state["q"])
        ring.wait()
        off, vals = ring.results()
        return off, _padded(vals, nq * KEYS)
    ring.submit_resident(nq)
    ring.wait()
    return _device_lists(ring)


# ------------------------------------------------------------------ cost model

N_IN, N_HID, N_OUT = tm.UNIT_FEATURES, 64, 3


def _mlp_data(case, seed):
    """Parameters, unit features in [0, 1) and log-scaled targets, float32."""
    rng = np.random.default_rng(seed)

    def layer(a, b):
        return [(rng.standard_normal((a, b)) * np.sqrt(2.0 / a)).ravel(), rng.standard_normal(b) * 0.05]

    p = np.concatenate(layer(N_IN, N_HID) + layer(N_HID, N_HID) + layer(N_HID, N_OUT)).astype(np.float32)
    x = rng.random((case["rows"], N_IN), np.float32)
    t = np.log2(1.0 + rng.lognormal(4.0, 3.0, (case["rows"], N_OUT))) / 16.0
    return p, x, t.astype(np.float32)


def _prepare_mlp(case, seed):
    tm.init(0)
    p, x, t = _mlp_data(case, seed)
    mlp = tm.MLP(N_IN, N_HID, N_OUT)
    mlp.set_params(p)
    return {"kind": "mlp", "mlp": mlp, "x": x, "t": t}


def exact(case, seed):
    if case["kind"] != "mlp":
        return None   # whole numbers throughout
    p, x, t = (a.astype(np.float64) for a in _mlp_data(case, seed))
    cut = np.cumsum([N_IN * N_HID, N_HID, N_HID * N_HID, N_HID, N_HID * N_OUT])
    w1, b1, w2, b2, w3, b3 = np.split(p, cut)
    w1, w2, w3 = w1.reshape(N_IN, N_HID), w2.reshape(N_HID, N_HID), w3.reshape(N_HID, N_OUT)
    h1 = np.maximum(x @ w1 + b1, 0.0)
    h2 = np.maximum(h1 @ w2 + b2, 0.0)
    d = h2 @ w3 + b3 - t
    loss = float(np.mean(d * d))
    dy = 2.0 * d / d.size
    d2 = (dy @ w3.T) * (h2 > 0)
    d1 = (d2 @ w2.T) * (h1 > 0)
    g = [x.T @ d1, d1.sum(0), h1.T @ d2, d2.sum(0), h2.T @ dy, dy.sum(0)]
    return loss, np.concatenate([a.ravel() for a in g])


# ------------------------------------------------------------------ work

def work(case):
    """Inputs read once and results written once.  Of the table, a step
    cannot do without the block masks (32 bytes for 64 filters), nor, where
    it lists matches or matches thousands of queries, without the filters and
    their key slots (32 bytes each)."""
    kind = case["kind"]
    if kind == "mlp":
        n = case["rows"]
        par = N_IN * N_HID + N_HID * N_HID + N_HID * N_OUT
        return {"bytes": 4.0 * (n * (N_IN + N_OUT) + 2 * (par + 2 * N_HID + N_OUT)),
                "flops": 6.0 * n * par - 2.0 * n * N_IN * N_HID}
    f = case["filters"]
    if kind == "partition":
        return {"bytes": f * 24.0 + f * 4.0, "flops": 0.0}
    masks, table = f / 64 * 32.0, f * 32.0
    if kind == "units":
        # about 500 queries a batch on average, a partition for every 67k filters
        nq = case["rounds"] * max(1.0, f / 67_000.0) * 500.0
        return {"bytes": nq * 24.0 + table + nq * (8.0 + 4.0 * 236), "flops": 0.0}
    nq = case["queries"]
    out = {"keys": 8.0 + 4.0 * KEYS, "every": KEYS / 8.0, "serve": KEYS / 8.0, "static": KEYS / 8.0,
           "packed": 4.0 + 0.01 * KEYS / 8.0, "hits": 8.0 + 8e-4 * f * 4.0, "keys_all": 8.0 + 7e-3 * f * 4.0}[kind]
    listing = kind in ("every", "hits", "keys_all") or nq > 4096
    return {"bytes": nq * (24.0 + out) + masks + (table if listing else 0.0), "flops": 0.0}
