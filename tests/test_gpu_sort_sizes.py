"""The sorts of the bulk path at the sizes where they change form: one
workgroup's sort, the split into buckets with short and long tiles, the row
scan of its histogram; uniform keys, keys repeated past a sub-bucket's and a
bucket's room.  The keys must come back as the ascending hashes (sequenced
ones in request order within a hash), and the table must count every key, on
a table of many regions and on one of few.  Every test prints its case before
it touches the GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _hash(k, bits):
    """hash_64 under the mask of `bits` bits, on numpy uint64."""
    m = np.uint64((1 << bits) - 1)
    u = np.uint64
    with np.errstate(over="ignore"):
        k = (~k + (k << u(21))) & m
        k = k ^ (k >> u(24))
        k = ((k + (k << u(3))) + (k << u(8))) & m
        k = k ^ (k >> u(14))
        k = ((k + (k << u(2))) + (k << u(4))) & m
        k = k ^ (k >> u(28))
        return (k + (k << u(31))) & m


SIZES = [1, 2, 1023, 8191, 8192, 8193, 20000, (1 << 18) - 1, 1 << 18, (1 << 20) + 1]


@pytest.mark.parametrize("q", [21, 24])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("distinct", [None, 300, 1])
def test_plain_sort(gpu, oracle, q, n, distinct):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    print(f"case sort q={q} n={n} distinct={distinct}", flush=True)
    keys = oracle.splitmix64(n + q, n)
    if distinct:
        keys = keys[:distinct][np.arange(n) % min(n, distinct)]
    f = GQF(q)
    try:
        dk = to_device_u64(keys)
        f.bulk_insert(dk)
        torch.cuda.synchronize()
        h = _hash(keys, q + 8)
        assert np.array_equal(to_numpy_u64(dk), np.sort(h))
        u, inv, cnt = np.unique(h, return_inverse=True, return_counts=True)
        got = to_numpy_u64(f.bulk_get(to_device_u64(keys)))
        assert np.array_equal(got, cnt[inv].astype(np.uint64))
        assert f.status() == 0 and f.layout_errors() == 0
        assert f.stats()["nelts"] == n and f.stats()["ndistinct_elts"] == u.size
    finally:
        f.close()


@pytest.mark.parametrize("q", [12, 22])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("distinct", [None, 300])
def test_sequenced_sort(gpu, oracle, q, n, distinct):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    print(f"case sequenced sort q={q} n={n} distinct={distinct}", flush=True)
    if q == 12 and (not distinct and n > 3000):
        n = 3000  # what the table holds
    keys = oracle.splitmix64(n + q, n)
    if distinct:
        keys = keys[:distinct][np.arange(n) % min(n, distinct)]
    nreq = min(n, 200)
    ends = sorted({(i + 1) * n // nreq for i in range(nreq)})
    seqs = [3 * i for i in range(len(ends))]
    dele = [i % 3 == 2 for i in range(len(ends))]
    f = GQF(q)
    try:
        dk = to_device_u64(keys)
        f.mutate_seq(dk, ends, [s << 1 | d for s, d in zip(seqs, dele)])
        torch.cuda.synchronize()
        h = _hash(keys, q + 8)
        req = np.searchsorted(np.array(ends), np.arange(n), side="right")
        tag = np.array([s | d << 15 for s, d in zip(seqs, dele)], dtype=np.uint64)[req]
        order = np.argsort(h, kind="stable")
        assert np.array_equal(to_numpy_u64(dk), (h | tag << np.uint64(48))[order])
        count = {}
        if n <= 20000:
            for x, d in zip(h.tolist(), np.array(dele)[req].tolist()):
                count[x] = max(0, count.get(x, 0) + (-1 if d else 1))
            got = to_numpy_u64(f.bulk_get(to_device_u64(keys)))
            assert np.array_equal(got, np.array([count[x] for x in h.tolist()], dtype=np.uint64))
        assert f.status() == 0 and f.layout_errors() == 0
    finally:
        f.close()
