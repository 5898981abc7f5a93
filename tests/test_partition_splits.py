"""The partitioner's kernels at the sizes where they can go wrong: tables cut
only by nonzero-mask splits around one workgroup's chunks (4096 filters) and
above what it takes at once (256k), balanced levels around the tiles of 1024,
sorted and shuffled tables.  Permutation, offsets and masks equal the
oracle's."""
import numpy as np
import pytest

import oracle as orc
import tagmatch_amd as tm

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 1), (192, 1 << 30), (1023, 1 << 30), (1025, 1 << 30), (4095, 1 << 30), (4097, 1 << 30),
         (20000, 1 << 30), (270000, 1 << 30), (1025, 1000), (2049, 300), (5000, 7), (30000, 1024)]


@pytest.mark.parametrize("n,maxp", SIZES)
def test_partition_splits_vs_oracle(gpu, n, maxp):
    words, _, _ = tm.canonicalize(*tm.Generator(seed=41).filters(n + n // 5 + 1))
    words = np.ascontiguousarray(words[:n])
    for order in (np.arange(n), np.random.default_rng(n).permutation(n)):
        w = np.ascontiguousarray(words[order])
        rc, perm, off, masks = orc.partition(w, maxp)
        assert rc == 0
        p, o, m = tm.partition(w, maxp)
        assert np.array_equal(p, perm) and np.array_equal(o, off) and np.array_equal(m, masks)


def test_single_bit_filters(gpu):
    """192 filters of one bit each: 191 splits of equal frequencies in a row."""
    w = np.zeros((192, 6), np.uint32)
    w[np.arange(192), np.arange(192) // 32] = np.uint32(1) << (np.arange(192) % 32).astype(np.uint32)
    rc, perm, off, masks = orc.partition(w, 1000)
    p, o, m = tm.partition(w, 1000)
    assert rc == 0 and np.array_equal(p, perm) and np.array_equal(o, off) and np.array_equal(m, masks)
