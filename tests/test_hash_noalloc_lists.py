"""The no-allocation table build where a bucket overflows its list of 32 pairs, after a build
of another size has left its own words in the shared scratch.  Pairs that a full bucket turns
away ask the overfull bucket for room in the next round, before the host learns that the table
is to be built by sorting: they must not be placed by what an earlier build left there."""
import numpy as np
import pytest
from sklearn.utils import murmurhash3_32 as sk_murmur

from oracle.pyoracle import HashOracle
from tests.test_hash import _coords, _random_keys

DIM, MAX_KEYS, GUARD = (128, 128, 128), 50000, 4096


def _murmur(c, seed):
    """MurmurHash3_x86_32 of each row of an (n, 3) int32 array."""
    def rot(v, r):
        return (v << np.uint32(r)) | (v >> np.uint32(32 - r))

    with np.errstate(over="ignore"):
        h = np.full(c.shape[0], seed, np.uint32)
        for a in range(3):
            k = rot(c[:, a].astype(np.uint32) * np.uint32(0xCC9E2D51), 15) * np.uint32(0x1B873593)
            h = rot(h ^ k, 13) * np.uint32(5) + np.uint32(0xE6546B64)
        h ^= np.uint32(12)
        h = (h ^ (h >> np.uint32(16))) * np.uint32(0x85EBCA6B)
        h = (h ^ (h >> np.uint32(13))) * np.uint32(0xC2B2AE35)
        return h ^ (h >> np.uint32(16))


def _spilling_keys(oracle, overfull, pairs):
    """`pairs` groups of keys: `overfull` of one round-0 bucket, and 17 of another, the largest
    of which asks the first for room in round 1."""
    allk = np.arange(np.prod(DIM), dtype=np.uint32)
    c = _coords(allk, DIM)
    b0, b1 = (_murmur(c, s) % np.uint32(oracle.buckets) for s in oracle.seeds[:2])
    for i in (0, 12345, 2000000):
        assert int(b1[i]) == sk_murmur(c[i].tobytes(), seed=int(oracle.seeds[1]), positive=True) % oracle.buckets
    groups, used = [], set()
    for full in range(oracle.buckets):
        # an asking key with at least 16 smaller ones in its own bucket
        for k in allk[b1 == full]:
            home = int(b0[k])
            small = allk[(b0 == home) & (allk < k)]
            if home == full or {home, full} & used or small.shape[0] < 16:
                continue
            groups.append(np.concatenate([allk[b0 == full][:overfull], small[:16], [k]]))
            used |= {home, full}
            break
        if len(groups) == pairs:
            return np.concatenate(groups).astype(np.uint32)
    raise AssertionError("too few groups")


def _build(keys, vals, max_keys=MAX_KEYS):
    import torch
    from ckmpm_amd.hashtable import build_noalloc, table_sizes

    ns, nt = table_sizes(max_keys)
    dk, dv = (torch.from_numpy(a.view(np.int32)).cuda() for a in (keys, vals))
    table = torch.full((GUARD + ns + GUARD + nt + GUARD,), -7, dtype=torch.int64, device="cuda")
    count = torch.full((1,), 99, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    at = table.data_ptr()
    rc = build_noalloc(DIM, max_keys, dk.data_ptr(), dv.data_ptr(), keys.shape[0], at + 8 * GUARD,
                       at + 8 * (2 * GUARD + ns), count.data_ptr())
    got = table.cpu().numpy()
    for g in (got[:GUARD], got[GUARD + ns:2 * GUARD + ns], got[-GUARD:]):
        assert (g == -7).all()
    return rc, got[GUARD:GUARD + ns].view(np.uint64), got[2 * GUARD + ns:].view(np.uint64), int(count.cpu()[0])


@pytest.mark.gpu
@pytest.mark.parametrize("overfull", [33, 40])
def test_overfull_bucket_after_a_build_of_another_size(overfull):
    from ckmpm_amd import native

    o = HashOracle(DIM, MAX_KEYS)
    keys = _spilling_keys(o, overfull, 8)
    vals = np.arange(keys.shape[0], dtype=np.uint32) + 7
    big = _random_keys(DIM, 200003, 4)
    o.build(keys, vals)
    for _ in range(2):
        # 200,003 pairs: the fills of the smaller table lie among this build's bucket lists
        assert _build(big, big, 200003)[0] == native.OK
        rc, slots, stash, n = _build(keys, vals)
        assert rc == native.OK
        np.testing.assert_array_equal(slots, o.slots)
        assert n == o.nstash
        np.testing.assert_array_equal(stash[:n], o.stash[:n])


@pytest.mark.gpu
def test_many_copies_of_one_key_are_refused():
    from ckmpm_amd import native

    o = HashOracle(DIM, MAX_KEYS)
    keys = _spilling_keys(o, 1, 8)
    keys = np.concatenate([keys, np.repeat(keys[::18], 39)])  # 40 copies of each first key
    big = _random_keys(DIM, 200003, 4)
    assert _build(big, big, 200003)[0] == native.OK
    assert _build(keys, keys)[0] == native.ERR_INVALID
