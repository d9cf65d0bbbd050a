"""The list build of the block table where its bucket lists fill up: keys that all ask for
bucket 0 in every round, at a bucket's size, at the list's (32 entries) and beyond, where
the sort build takes over.  Slots and stash equal the oracle's, word for word."""
import numpy as np
import pytest

from oracle.pyoracle import HashOracle
from tests.test_hash import _random_keys, _stash_keys

DIM = (16, 16, 16)


@pytest.mark.gpu
@pytest.mark.parametrize("collide,others", [(1, 0), (16, 0), (17, 5), (32, 0), (32, 8), (33, 0), (33, 7), (40, 0)])
def test_gpu_lists_match_the_oracle(collide, others):
    from ckmpm_amd.hashtable import BlockHashTable

    o = HashOracle(DIM, 40)
    keys = _stash_keys(DIM, o.buckets, o.seeds, collide)
    keys = np.concatenate([np.setdiff1d(_random_keys(DIM, 80, 5), keys)[:others].astype(np.uint32), keys[::-1]])
    vals = np.arange(keys.shape[0], dtype=np.uint32) + 7
    o.build(keys, vals)
    g = BlockHashTable(DIM, 40)
    for _ in range(2):  # a rebuild of the same table starts from what the first one left
        g.Insert(keys, vals)
        slots, stash = g.export()
        np.testing.assert_array_equal(slots, o.slots)
        np.testing.assert_array_equal(stash, o.stash[:o.nstash])
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("collide", [3, 40])
def test_gpu_lists_refuse_what_the_sort_refuses(collide):
    from ckmpm_amd.hashtable import BlockHashTable
    from ckmpm_amd.native import CkmpmError

    o = HashOracle(DIM, 40)
    keys = _stash_keys(DIM, o.buckets, o.seeds, collide)
    dup, bad = keys.copy(), keys.copy()
    dup[-1] = dup[0]
    bad[1] = 16 ** 3
    g = BlockHashTable(DIM, 40)
    vals = np.arange(collide, dtype=np.uint32)
    for k, msg in ((dup, "duplicate"), (bad, "outside the domain")):
        with pytest.raises(CkmpmError, match=msg):
            g.Insert(k, vals)
    g.Insert(keys, vals)
    np.testing.assert_array_equal(g.Find(keys), vals)
    g.close()
