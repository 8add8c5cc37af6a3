"""Batches that a table cannot hold: the filter has to say so, its layout
stays sound, what was in it stays, and a region (48 blocks of quotients) takes
all of its new items or none.  More regions overflow here than the wide pass
lists, so its classes redo them.  Prints its case before it touches the
GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["insert", "requests"])
@pytest.mark.parametrize("extra", [0.08, 0.4])
def test_regions_whole_or_not(gpu, oracle, how, extra):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    q = 20
    print(f"case full table {how} {extra}", flush=True)
    rng = np.random.default_rng(int(100 * extra))
    hs = np.unique(rng.integers(0, 1 << (q + 8), size=3 << q, dtype=np.uint64))
    rng.shuffle(hs)
    n0, n1 = int(0.9 * (1 << q)), int(extra * (1 << q))
    old, new = hs[:n0], hs[n0:n0 + n1]
    f = GQF(q)
    try:
        f.bulk_insert(to_device_u64(old), flags=0x08)
        torch.cuda.synchronize()
        assert f.status() == 0
        if how == "insert":
            f.bulk_insert(to_device_u64(new), flags=0x08)
        else:
            keys = np.array([oracle.hash_64i(int(h), (1 << (q + 8)) - 1) for h in new], dtype=np.uint64)
            f.mutate_seq(to_device_u64(keys), [n1 // 2, n1], [0, 2])
        torch.cuda.synchronize()
        assert f.layout_errors() == 0
        hashes, counts = (to_numpy_u64(x) for x in f.enumerate())
        assert (counts == 1).all() and np.isin(old, hashes).all()
        region = (new >> np.uint64(14)) // np.uint64(f.info["region_blocks"])
        there = np.isin(new, hashes)
        n = np.bincount(region.astype(np.int64))
        got = np.bincount(region.astype(np.int64), weights=there).astype(np.int64)
        assert ((got == 0) | (got == n)).all()
        assert hashes.size == n0 + int(there.sum())
        assert there.all() or f.status() != 0
        assert extra < 0.2 or not there.all()
    finally:
        f.close()
