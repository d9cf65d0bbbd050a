"""The list build of the smallest block tables: one to three buckets, where the lists take the
most words per pair of the table's capacity."""
import numpy as np
import pytest

from oracle.pyoracle import HashOracle
from tests.test_hash import _random_keys

DIM = (16, 16, 16)


@pytest.mark.gpu
@pytest.mark.parametrize("max_keys", [1, 2, 11, 12, 23])
def test_gpu_lists_of_the_smallest_tables(max_keys):
    from ckmpm_amd.hashtable import BlockHashTable

    keys = _random_keys(DIM, max_keys, max_keys)
    vals = keys ^ np.uint32(0x55)
    o = HashOracle(DIM, max_keys)
    o.build(keys, vals)
    g = BlockHashTable(DIM, max_keys)
    g.Insert(keys, vals)
    slots, stash = g.export()
    np.testing.assert_array_equal(slots, o.slots)
    np.testing.assert_array_equal(stash, o.stash[:o.nstash])
    np.testing.assert_array_equal(g.Find(keys), vals)
    g.close()
