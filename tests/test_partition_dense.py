"""Nonzero-mask splits of filters with many bits set, which the partitioner
makes level by level down to half a million set bits and then in one
workgroup: around that count, with the filter of every bit among them.
Permutation, offsets and masks equal the oracle's."""
import time

import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu


def filters(n, density, seed):
    b = np.random.default_rng(seed).random((n, 192)) < density
    w = np.ascontiguousarray(np.packbits(b, axis=1, bitorder="little").view(np.uint32))
    w[n // 2] = 0xFFFFFFFF
    w[~w.any(axis=1), 5] = 1      # (the oracle takes no empty filter)
    return w


@pytest.mark.parametrize("n,density", [(2604, 1.0), (2605, 1.0), (5000, 0.5), (5400, 0.5), (40000, 0.5), (40000, 0.1),
                                       (60000, 0.02)])
@pytest.mark.parametrize("maxp", [3000, 1 << 30])
def test_dense_splits_vs_oracle(gpu, n, density, maxp):
    w = filters(n, density, n)
    rc, perm, off, masks = orc.partition(w, maxp)
    assert rc == 0
    p, o, m = tm.partition(w, maxp)
    assert np.array_equal(p, perm) and np.array_equal(o, off) and np.array_equal(m, masks)


def test_dense_splits_take_no_longer_than_levels(gpu):
    """200k filters with half their bits set: one nonzero-mask segment, at
    most three times as long as balanced levels down to 8192 filters."""
    w = filters(200_000, 0.5, 1)
    best = []
    for maxp in (1 << 30, 8192):
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            tm.partition(w, maxp)
            t.append(time.perf_counter() - t0)
        best.append(min(t))
    print(f"ms {[1e3 * x for x in best]}", flush=True)
    assert best[0] < 3 * best[1]
