"""The counting reduce's buckets, by the hash's top bits: from one distinct
hash to several thousand in a bucket, at hash widths on both sides of the
bucket bits' and key widths that leave value bits, against numpy: the keys left
sorted, every count, and the table's totals.  Prints its case before it
touches the GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# n at least 2^22 with fewer than half of a sample distinct, which the counting takes
@pytest.mark.parametrize("q,distinct,rest", [(10, 1, 0), (12, 3, 0), (16, 511, 0), (18, 513, 100), (20, 1500, 700),
                                             (22, 300, 60000), (24, 300, 1900000), (32, 300, 70000)])
def test_count_buckets(gpu, oracle, q, distinct, rest):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    n = (1 << 22) + 77
    print(f"case count q={q} distinct={distinct} rest={rest}", flush=True)
    ids = oracle.splitmix64(q, distinct + rest)
    draw = oracle.splitmix64(q + 1, n)
    pick = draw % np.uint64(distinct)
    if rest:  # two in five draws from the rest
        pick = np.where((draw >> np.uint64(40)) % np.uint64(5) < 2,
                        np.uint64(distinct) + (draw >> np.uint64(8)) % np.uint64(rest), pick)
    keys = ids[pick.astype(np.int64)]
    f = GQF(q)
    try:
        dk = to_device_u64(keys)
        f.bulk_insert_reduce(dk)
        torch.cuda.synchronize()
        assert f.status() == 0 and f.layout_errors() == 0
        h = to_numpy_u64(dk)
        assert (h[1:] >= h[:-1]).all()
        u, cnt = np.unique(h, return_counts=True)
        hashes, counts = f.enumerate()
        assert np.array_equal(to_numpy_u64(hashes), u)
        assert np.array_equal(to_numpy_u64(counts), cnt.astype(np.uint64))
        # the hashes are those of the keys: each key's count is that of its copies
        k, inv, kc = np.unique(keys & np.uint64((1 << (q + 8)) - 1), return_inverse=True, return_counts=True)
        got = to_numpy_u64(f.bulk_get(to_device_u64(k)))
        assert np.array_equal(got, kc.astype(np.uint64))
    finally:
        f.close()
